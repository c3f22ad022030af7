"""The selection of one row by sixteen waves must not depend on how far one of them is ahead of another between two barriers:
the kernel's own text, on the CPU, with the waves in chosen orders (tests/native/select_few_waves.cpp), against a
stable sort of the keys."""
import numpy as np
import pytest

from tests.util import select_few_waves


def keys_of(x, total_order):
    x = np.ascontiguousarray(x if total_order else np.where(x == 0, np.float32(0), x), np.float32)
    b = x.view(np.uint32)
    return (b ^ np.where(b >> 31, np.uint32(0xFFFFFFFF), np.uint32(0x80000000))).astype(np.int64)


def rows_of(nt):
    """One value (no histogram), one value with NaNs of the lowest key, few values (histograms refined to a bin of equal keys), a
    narrow range between outliers (refined more than once), spread."""
    rng = np.random.default_rng(nt)
    yield np.zeros(nt, np.float32)
    x = np.full(nt, 2.5, np.float32)
    x.view(np.uint32)[[0, nt // 2, nt - 1]] = 0xFFFFFFFF
    yield x
    yield rng.integers(0, 3, nt).astype(np.float32)
    x = (1 + rng.random(nt) * 1e-3).astype(np.float32)
    x[0], x[-1] = 3e38, -3e38
    yield x
    yield rng.standard_normal(nt).astype(np.float32)


@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("nt", [65, 1000, 2048, 5000, 16384])
def test_the_order_of_the_waves_does_not_matter(nt, order):
    for r, x in enumerate(rows_of(nt)):
        for total_order in (False, True):
            keys = keys_of(x, total_order)
            for k in (nt // 3, nt - 1):
                want = np.sort(np.argsort(-keys, kind="stable")[:k]) + 128
                got = select_few_waves(x, k, total_order, 128, order)
                assert got is not None and np.array_equal(got, want), (r, k, total_order)
