"""The selection of one row by one workgroup with the keys in registers (up to 16 384 scores), through both entry
points that use it: the row selection (-0.0 equal to +0.0) and the block selection (IEEE total order), against a
stable sort of the keys. Whole numbers, so exact."""
import numpy as np
import pytest

from rivoli_amd import hip
from tests.gpu_util import back, dev, dzeros

pytestmark = pytest.mark.gpu


def total_order(x):
    b = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return b ^ np.where(b >> 31, np.uint32(0xFFFFFFFF), np.uint32(0x80000000))


def want_rows(keys, k):
    order = np.argsort(-keys.astype(np.int64), kind="stable")[:k]
    return np.sort(order)


def rows_of(nt, rng):
    """Distributions that place the pivot differently: spread, a narrow range, a range stretched by outliers, few values,
    one value, the type's lowest value over most of a row, sparse, rounded to bf16, zeros of both signs."""
    n = rng.standard_normal(nt).astype(np.float32)
    yield n
    yield (1 + rng.random(nt) * 1e-5).astype(np.float32)
    x = (1 + rng.random(nt) * 1e-3).astype(np.float32)
    x[0], x[-1] = 3e38, -3e38
    yield x
    yield rng.integers(0, 3, nt).astype(np.float32)
    yield np.full(nt, -2.5, np.float32)
    x = np.abs(n) + 1
    x[nt // 3:] = np.finfo(np.float32).min
    yield x
    yield np.maximum(n - 1.5, 0).astype(np.float32)
    yield (n.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    yield (rng.integers(-1, 2, nt) * np.float32(0.0)).astype(np.float32)
    x = n.copy()
    x[:2], x[-1] = -np.inf, np.inf
    yield x


@pytest.mark.parametrize("nt", [2, 63, 65, 1024, 1025, 2048, 2049, 4097, 8192, 8193, 16384])
def test_selection_of_one_row(nt):
    rng = np.random.default_rng(nt)
    rows = np.stack(list(rows_of(nt, rng)))
    for k in sorted({1, 2, min(512, nt - 1), nt - 1, nt}):
        keys = total_order(np.where(rows == 0, np.float32(0), rows))
        d_rows = dzeros(len(rows) * k * 4, 0xEE)
        hip.launch_index_topk_batched(dev(rows), len(rows), nt, None, nt, k, d_rows, None)
        got = back(d_rows, np.int32).reshape(len(rows), k)
        for r in range(len(rows)):
            assert np.array_equal(got[r], want_rows(keys[r], k)), (nt, k, r)
    if nt <= 512:
        return
    blocks = rows.copy()
    for r, bits in ((0, 0xFFFFFFFF), (2, 0xFFC00000), (3, 0x7FC00001)):  # the first is the lowest key there is, 0
        b = blocks[r].view(np.uint32)
        b[[1, nt // 2, nt - 1]] = bits
    keys = total_order(blocks)
    for k in (1, 512, min(nt - 1, 4000)):
        d_out = dzeros(len(rows) * k * 4, 0xEE)
        hip.launch_index_select_blocks(dev(blocks), len(rows), nt, 4, k, False, 128, d_out)
        got = back(d_out, np.int32).reshape(len(rows), k)
        for r in range(len(rows)):
            assert np.array_equal(got[r], want_rows(keys[r], k) + 128), (nt, k, r)
    # all but one of a row taken, its lowest key among them more than once
    k = nt - 1
    d_out = dzeros(len(rows) * k * 4, 0xEE)
    hip.launch_index_select_blocks(dev(blocks), len(rows), nt, 4, k, False, 0, d_out)
    got = back(d_out, np.int32).reshape(len(rows), k)
    for r in range(len(rows)):
        assert np.array_equal(got[r], want_rows(keys[r], k)), (nt, k, r)
