"""Host-side restatement of the index arithmetic of the block scorer's head-split kernel
(rivoli_amd/csrc/block_index.hip: index_score_blocks_128_split_kernel + walk_pairs): which
floats of q a wave requests, for head counts that leave some of the eight waves without a head.
Every request must stay inside q[s][heads][128]; a wave without heads requests nothing. And the rule by which a call takes its
kernel and its grid (block_index_plan.hpp)."""
import pytest

import bench
from tests.util import score_plan

WAVES, HD, CHUNK = 8, 128, 32


def wave_requests(s, heads, wave, t, guard=True):
    """(first, last) float offsets of every chunk the wave requests for query t."""
    per = -(-heads // WAVES)
    h0 = min(wave * per, heads)
    h1 = min(h0 + per, heads)
    g0, g1 = t * heads + h0, t * heads + h1
    if guard and g0 >= g1:
        return []
    out = []
    qp = g0 * HD
    out.append((qp, qp + CHUNK - 1))                      # the first chunk, before the loop
    for g in range(g0, g1):
        for off in (32, 64, 96):
            out.append((qp + off, qp + off + CHUNK - 1))
        nxt = qp + HD if g + 1 < g1 else qp               # the next pair's first chunk, or its own again
        out.append((nxt, nxt + CHUNK - 1))
        qp += HD
    return out


@pytest.mark.parametrize("heads", [1, 2, 5, 7, 8, 9, 11, 17, 20, 63, 64, 65, 128])
@pytest.mark.parametrize("s", [1, 2, 65])
def test_every_request_stays_inside_q(s, heads):
    size = s * heads * HD
    covered = set()
    for t in range(s):
        for wave in range(WAVES):
            for first, last in wave_requests(s, heads, wave, t):
                assert 0 <= first and last < size, (s, heads, wave, t, first, last, size)
                covered.update(range(first // CHUNK, last // CHUNK + 1))
    assert covered == set(range(size // CHUNK))           # and every chunk of q is read by someone


def test_a_wave_without_heads_would_read_past_the_end_without_the_guard():
    s, heads = 2, 5                                       # per = 1: waves 5..7 have no head
    size = s * heads * HD
    assert wave_requests(s, heads, 7, s - 1) == []
    first, last = wave_requests(s, heads, 7, s - 1, guard=False)[0]
    assert last >= size                                   # what the guard is there for


def test_the_scorers_grid_covers_its_blocks_and_the_benchmark_names_its_kernel():
    """Every block is one workgroup's, splits are whole tiles that a 128-bit mask holds, and bench.block_scorer is the launcher's rule."""
    seen = set()
    for s in (1, 2, 3, 7, 8, 9, 16, 17, 100, 104, 300, 384, 385, 700, 1024, 1500, 2049, 3000, 4096, 6001, 8191, 8192, 8193, 32768, 2 ** 20):
        for n_comp in (1, 2, 31, 32, 33, 63, 64, 65, 75, 128, 175, 191, 192, 193, 375, 512, 750, 1024, 2048, 4096, 4097, 8192, 65536, 2 ** 20):
            kernel, split, groups, rows = score_plan(s, n_comp)
            seen.add(kernel)
            name = {"one 32": "score_blocks_one_kernel", "one 64": "score_blocks_one_kernel", "pair": "score_blocks_pair_kernel",
                    "codes": "score_blocks_codes_kernel"}[kernel]
            assert bench.block_scorer(s, n_comp)[0] == name, (s, n_comp)
            assert (s == 1 or s * -(-n_comp // 64) <= 384) == kernel.startswith("one")
            if not kernel.startswith("one"):
                assert groups * 8 >= s > (groups - 1) * 8 and split % 32 == 0 and 32 <= split <= 4096
                assert rows * split >= n_comp > (rows - 1) * split and rows <= 65535
                assert kernel == "pair" or split >= 192 or split == 32
    assert seen == {"one 32", "one 64", "pair", "codes"}
    # the lines, on both sides
    assert [score_plan(s, n)[0] for s, n in ((2049, 512), (1500, 375), (4, 4096), (4, 8192), (1, 16384), (1, 8192))] == \
        ["codes", "pair", "one 64", "pair", "one 64", "one 32"]
