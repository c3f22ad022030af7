"""The launchers' Python functions (csrc/pylaunch.cpp): one per status-returning entry point of the
header, with its argument count, and each kind of argument converted or refused."""
import ctypes as C
import re

import pytest
import torch

from rivoli_amd import hip
from tests.test_abi_drift import header_prototypes


def test_one_function_per_entry_point_with_its_argument_count():
    for sym, (ret, args) in header_prototypes().items():
        if ret == "usize":
            continue
        with pytest.raises(TypeError) as e:
            getattr(hip.entry, sym)(*([None] * (len(args) + 1)))
        assert re.match(rf"{len(args)} arguments expected, {len(args) + 1} given", str(e.value)), sym
    with pytest.raises(AttributeError):
        hip.entry.rivoli_no_such_entry


def test_arguments_are_converted_by_kind():
    t = torch.zeros(64)
    call = hip.entry.rivoli_kv_append_paged
    ok = [t, t, t, 0, 576, 64, 10, None, None]           # no tokens: 1001 before anything is launched
    assert call(*ok) == 1001
    assert call(*(ok[:3] + [1, 1025] + ok[5:])) == 1002  # pointers arrived, the width guard answers
    assert call(*([None] + ok[1:3] + [1] + ok[4:])) == 1001
    # an address is taken as it is: 8 past an aligned one fails the alignment guard
    assert call(*([t.data_ptr() + 8 & ~7 | 8] + ok[1:3] + [1] + ok[4:])) == 1004
    for at, bad, error in ((0, "x", AttributeError), (0, 1.5, AttributeError), (3, 0.0, TypeError), (3, None, TypeError),
                           (8, t, AttributeError)):
        args = list(ok)
        args[at] = bad
        with pytest.raises(error):
            call(*args)

    class Stream:
        cuda_stream = 5

    assert call(*(ok[:8] + [Stream()])) == 1001
    rows, cols = C.c_int(0), C.c_int(0)
    assert hip.entry.rivoli_sel_shape(8, 4, 512, 2 ** 32 + 12, 0, C.addressof(rows), C.addressof(cols)) == 0
    assert (rows.value, cols.value) == (12, 11)          # an int narrows as C would
