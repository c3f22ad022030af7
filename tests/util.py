"""Seeded synthetic inputs shared by the oracle and GPU parity tests (numpy only)."""
import ctypes
import os
import subprocess

import numpy as np


def f32_to_bf16_rne(x: np.ndarray) -> np.ndarray:
    """Textbook integer round-to-nearest-even; finite inputs only."""
    b = np.ascontiguousarray(x, np.float32).view(np.uint32)
    # uint32 arithmetic cannot wrap for finite inputs (|bits| <= 0x7f7fffff before the add)
    r = (b >> np.uint32(16)) & np.uint32(1)
    r += np.uint32(0x7FFF)
    r += b
    r >>= np.uint32(16)
    return r.astype(np.uint16)


def bf16_to_f32(b: np.ndarray) -> np.ndarray:
    return (np.ascontiguousarray(b, np.uint16).astype(np.uint32) << 16).view(np.float32)


def make_rows_bf16(n, width=576, seed=0, outlier_frac=0.0, outlier_mul=1.0) -> np.ndarray:
    """[n, width] bf16 bit patterns: N(0,1) in f32, a fraction of ROWS scaled, then RNE to bf16.
    That bf16 tensor is the input both the oracle and the kernels receive."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, width), dtype=np.float32)
    if outlier_frac > 0:
        hit = rng.random(n) < outlier_frac
        x[hit] *= np.float32(outlier_mul)
    return f32_to_bf16_rne(x)


def shuffled_block_tables(n_seqs, blocks_per_seq, n_pages, seed):
    """Disjoint pages for every sequence, drawn from one shuffled global pool."""
    rng = np.random.default_rng(seed)
    perm = rng.permutation(n_pages).astype(np.int32)
    assert n_seqs * blocks_per_seq <= n_pages
    return perm[: n_seqs * blocks_per_seq].reshape(n_seqs, blocks_per_seq).copy()


def slots_for(table_row, positions, page_tokens=64):
    positions = np.asarray(positions)
    return (table_row[positions // page_tokens] * page_tokens + positions % page_tokens).astype(np.int32)


class AttendRoute:
    """attend_route of rivoli_amd/csrc/mla_attend_plan.hpp: which workgroups a call of the shipped row
    widths takes, and its work items; `few`: of 16 heads, with eight waves on a tile. `linear`: over the linear slabs, 1 with scratch, 2 without."""

    def __init__(self, heads16, out):
        self.heads16 = bool(heads16)
        self.items, self.by_seq, self.records, self.scratch_items, self.scratch_records, few = list(out)
        self.few = bool(few)


def _plan():
    global _PLAN
    if _PLAN is None:
        here = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")
        path = os.path.join(here, "attend_plan.so")
        if not os.path.exists(path):
            subprocess.run(["make", "-C", here, path], check=True, capture_output=True)
        _PLAN = ctypes.CDLL(path)
        _PLAN.marked_block.restype = ctypes.c_longlong
    return _PLAN


def attend_route(n_seqs, H, max_rows, precise, listed=False, linear=0):
    out = (ctypes.c_int * 6)()
    return AttendRoute(_plan().attend_route(n_seqs, H, max_rows, precise, int(listed), linear, out), out)


def attend_wide_items(n_seqs, H, max_rows, precise, listed=False):
    """heads32_route of the same file: a paged call's work items in workgroups of 32 heads, 0 where attend_route's route stands."""
    return _plan().attend_wide_items(n_seqs, H, max_rows, precise, int(listed))


def score_plan(s, n_comp):
    """rivoli_amd/csrc/block_index_plan.hpp: the block scorer's kernel for a call of 128 dims and up to 64 heads, blocks of a workgroup
    of the many-query kernels and their grid."""
    out = (ctypes.c_int * 3)()
    kernel = ("one 32", "one 64", "pair", "codes", "none")[_plan().score_plan(s, n_comp, out)]
    return (kernel, *out)


def marked_block(row, group):
    """rivoli_amd/csrc/gather_attn_plan.hpp: the group's block in a row of 256."""
    return _plan().marked_block(row, group)


_PLAN = None


_WAVES = None


def select_few_waves(scores, k, total_order, add, order):
    """The k best of a row by rivoli_amd/csrc/select_few.hpp on the CPU, its waves in the given order between two barriers
    (tests/native/select_few_waves.cpp); None where its barriers never end."""
    global _WAVES
    if _WAVES is None:
        here = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")
        path = os.path.join(here, "select_few_waves.so")
        if not os.path.exists(path):
            subprocess.run(["make", "-C", here, path], check=True, capture_output=True)
        _WAVES = ctypes.CDLL(path)
    scores = np.ascontiguousarray(scores, np.float32)
    items = next(i for i in (1, 2, 8, 16) if len(scores) <= 1024 * i)
    out = np.full(k, 0xEEEEEEEE, np.uint32)
    ended = _WAVES.select_few_waves(scores.ctypes.data_as(ctypes.c_void_p), len(scores), k, items, int(total_order),
                                    ctypes.c_uint32(add), order, out.ctypes.data_as(ctypes.c_void_p))
    return out if ended >= 0 else None
