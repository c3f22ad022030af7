"""Which kernel an attention call takes and how its tiles are shared
(rivoli_amd/csrc/mla_attend_plan.hpp, compiled for the host by tests/native/Makefile)."""
import numpy as np
import pytest

from tests.util import attend_route, attend_wide_items, marked_block


@pytest.mark.parametrize("listed", [False, True])
@pytest.mark.parametrize("precise", [0, 2, 4])
def test_a_plan_fits_the_scratch_and_the_chip(precise, listed):
    """Over head counts, batches and lengths: never more records than the caller's scratch was sized
    for, every work item with a tile a wave, and whole sequences where there is nothing to deal."""
    for H in (1, 16, 17, 33, 48, 64, 80, 128, 200, 528, 4096):
        for n in (1, 2, 7, 16, 33, 64, 65, 100, 128, 129, 200, 255, 256, 1024, 1025, 5000):
            for rows in (1, 32, 33, 64, 255, 256, 300, 512, 1000, 1984, 4096, 40000, 2 ** 25):
                r = attend_route(n, H, rows, precise, listed)
                tiles = -(-rows // 32)
                if not r.heads16:
                    assert r.items == r.scratch_items and r.records == r.scratch_records
                    continue
                assert r.items <= r.scratch_items and r.records <= r.scratch_records
                assert r.records == (r.items + n if r.items else 0)
                groups = -(-H // 16)    # the groups of an item sit on one of the eight dies of 32 units
                assert groups > 32 or -(-r.items // 8) * groups <= 32, (H, n, rows, r.items)
                assert r.items == 0 or (r.items >= n and r.items <= n * (tiles // 4))
                assert not r.by_seq or (n <= 64 and r.items >= 2 * n)


@pytest.mark.parametrize("precise", [2, 4])
def test_batches_of_short_sequences_keep_to_the_kernel_of_fewer_rounds(precise):
    """Sequences that stay whole are a workgroup for every 16 heads in one kernel and for every 64 in
    the other: where the first need more rounds of the 256 compute units, short calls are the
    other's (128 sequences of 128 tokens at 128 heads: four rounds against one)."""
    for H, n in ((128, 64), (128, 128), (64, 128), (64, 256), (32, 256), (48, 85), (80, 51)):
        for rows in (32, 64, 128, 256, 320):
            for listed in (False, True):
                assert not attend_route(n, H, rows, precise, listed).heads16, (H, n, rows)
    for H, n in ((128, 32), (64, 64), (32, 128), (16, 256), (48, 80), (80, 48)):
        assert attend_route(n, H, 128, precise).heads16, (H, n)
    # one round more is made good where the other kernel splits
    assert attend_route(128, 64, 512, 2).heads16 and not attend_route(34, 128, 960, 2).heads16
    assert attend_route(136, 32, 960, 2).heads16 and not attend_route(128, 64, 512, 4).heads16
    # nothing for most of the four waves to do
    for H, rows in ((16, 1), (16, 64), (32, 33), (64, 1), (128, 32)):
        assert attend_route(4, H, rows, precise).heads16 == (precise == 4), (H, rows)
    assert attend_route(4, 32, 64, 2, listed=True).heads16 and attend_route(4, 64, 64, 2).heads16
    # three tiles of a second round of few-head sequences: the other's where most are shorter than that
    for n, rows, there in ((256, 96, True), (257, 96, False), (257, 97, True), (1000, 65, False), (1000, 128, True)):
        assert attend_route(n, 16, rows, precise).heads16 == (there or precise == 4), (n, rows)


@pytest.mark.parametrize("precise", [0, 2])
def test_no_batch_of_long_sequences_is_left_whole(precise):
    """Past 32 tiles the lengths may differ widely, and the host does not know them: whichever kernel
    takes such a call deals its tiles out, also with fewer than two work items a sequence (129 to 255
    sequences of 16 heads, where one of 32 768 tokens took 769 us on a workgroup of its own)."""
    for H in (8, 16, 17, 32, 64, 96, 128):
        for n in list(range(1, 256, 6)) + [128, 129, 200, 254, 255]:
            for rows in (1025, 1984, 4096, 32768):
                r = attend_route(n, H, rows, precise)
                # (whole only where there is no scratch to merge from, or the other kernel's splits are
                # more than a round of workgroups themselves)
                assert r.items or not r.scratch_items or (r.scratch_items * -(-H // 64) > 256 and H > 16 and rows < 2048), \
                    (H, n, rows)


def test_calls_of_more_head_groups_than_a_die_has_units_stay_with_the_other_kernel():
    """Past 512 heads the groups of one work item are more than the 32 units of the die they sit on: a
    call of 2 048 heads took twice its time so. The linear slabs' other kernel is slow enough for two
    rounds of them over few rows."""
    for rows in (64, 512, 1024, 2048, 4096, 40000):
        for n in (1, 2, 7):
            for precise in (0, 2, 4):
                for listed in (False, True):
                    assert not any(attend_route(n, H, rows, precise, listed).heads16 for H in (513, 768, 1024, 2048, 8192))
        for linear in (1, 2):
            assert not any(attend_route(1, H, rows, 2, linear=linear).heads16 for H in (1025, 1536, 2048, 8192))
    for H in (520, 768, 1024):
        assert all(attend_route(1, H, rows, 2, linear=1).heads16 for rows in (512, 1024, 2048))
        assert not attend_route(1, H, 2049, 2, linear=1).heads16
    for linear in (1, 2):                   # ... and for any number of rows where the groups fit
        assert all(attend_route(1, H, rows, 2, linear=linear).heads16
                   for H in (1, 17, 64, 128, 512) for rows in (1, 300, 20000, 65537, 2 ** 24))
    assert attend_route(1, 512, 2048, 2).heads16 and attend_route(1, 512, 2048, 4, listed=True).heads16


@pytest.mark.parametrize("r_end", [1, 33, 2 ** 20, 2 ** 31 - 400, 2 ** 31 - 32])
def test_list_positions_looked_up_ahead_stay_in_the_list(r_end):
    """Host-side restatement of token_of in mla_attend_heads16.hpp: which list entries a wave asks for
    while it walks every fourth tile and looks up three of its own ahead. In 32 bits, unsigned; as
    ints the last rounds of the longest lists would wrap to entries in front of the list."""
    def wrapped(x, signed):
        x &= 0xFFFFFFFF
        return x - 2 ** 32 if signed and x >= 2 ** 31 else x

    n_tiles = -(-r_end // 32)
    for wave in range(4):
        last = wave + (n_tiles - 1 - wave) // 4 * 4 if n_tiles > wave else wave
        for tile in {wave, wave + 4, wave + 8, last, last + 4, last + 8, last + 12}:
            for lane in (0, 31):
                assert min(wrapped(tile * 32 + lane, False), r_end - 1) in range(r_end)
    if r_end > 2 ** 31 - 384:
        assert min(wrapped((n_tiles + 11) * 32, True), r_end - 1) < 0


def test_which_calls_of_16_heads_a_workgroup_share_a_tile_among_eight_waves():
    """All with three groups of heads, all over the linear slabs, and short work items: 48 tiles of 32 listed rows; of dense
    ones 56 where sequences stay whole, 96 where work items share them evenly, 128 where no item meets two of them; where
    q and weights are carried once, 96 and 64."""
    for rows in (64, 512, 4096, 40000):
        for H in (33, 64, 512):
            r = attend_route(1, H, rows, 2)
            assert r.few == r.heads16
        for linear in (1, 2):
            assert all(attend_route(1, H, rows, 2, linear=linear).few for H in (1, 16, 32, 64, 512))
    for precise, whole, shared, cut in ((2, 56, 96, 128), (1, 56, 96, 128), (0, 96, 64, 64)):
        for n, rows, tiles, listed in ((300, 32 * whole, whole, False), (300, 32 * 48, 48, True), (1, 32 * cut * 64, cut, False),
                                       (200, 32 * shared, shared, False),
                                       (64, 32 * cut * 4, cut, False), (64, 32 * 48 * 4, 48, True), (1, 32 * 48 * 64, 48, True)):
            at, past = attend_route(n, 16, rows, precise, listed), attend_route(n, 16, rows + 32 * 64, precise, listed)
            assert at.heads16 and at.few and past.heads16 and not past.few, (precise, n, rows, listed)
            assert not at.items or -(-n * -(-rows // 32) // at.items) == tiles


def test_blocks_left_to_a_second_pass_spread_over_its_groups():
    """The index-list attention's second pass: every block is one group's, all blocks are dealt evenly, and of blocks at
    any regular distance (a remainder in every 256th query) the fullest group has a few more than its share, not all."""
    rows = 32
    owner = np.full(rows * 256, -1)
    for row in range(rows):
        for group in range(256):
            block = marked_block(row, group)
            assert block // 256 == row and owner[block] == -1
            owner[block] = group
    assert marked_block(2 ** 24, 7) // 256 == 2 ** 24
    for stride in range(1, 2049):
        most = np.bincount(owner[::stride]).max()
        assert most <= -(-len(owner[::stride]) // 256) + 6, stride


@pytest.mark.parametrize("listed", [False, True])
@pytest.mark.parametrize("precise", [0, 2, 4])
def test_work_items_of_32_heads_fit_the_scratch_and_the_chip(precise, listed):
    """Never more records than the caller's scratch was sized for (an item and a sequence each), two work items a sequence and
    more, the head groups of all of them in one round of the compute units; and the calls that change sides."""
    for H in (1, 16, 17, 32, 33, 48, 64, 80, 128, 200, 528, 1024, 4096):
        for n in (1, 2, 7, 16, 20, 24, 33, 64, 65, 128, 1025):
            for rows in (1, 64, 300, 1000, 4096, 40000, 2 ** 25):
                items = attend_wide_items(n, H, rows, precise, listed)
                if not items:
                    continue
                assert H > 16 and n <= 64 and 2 * n <= items <= n * (-(-rows // 32) // 2), (H, n, rows, items)
                assert items <= attend_route(n, H, rows, precise, listed).scratch_items
                assert -(-items // 8) * 8 * -(-H // 32) <= 256
    wide = lambda *call: attend_wide_items(*call, precise, listed) > 0
    assert wide(24, 64, 8000) and wide(9, 128, 16384) and wide(18, 64, 10262)  # a second round of 64 heads' workgroups
    assert wide(6, 64, 9000) == (listed and precise < 4) and not wide(8, 64, 2048) and not wide(32, 64, 32768) and not wide(32, 16, 16384)
    assert wide(32, 64, 6000) == (precise < 4) and wide(12, 128, 2048) == (listed and precise < 4)


def test_work_items_of_32_heads_where_they_are_the_shorter_way():
    """Calls timed on both sides of the lines: the 8-bit modes' long ones and the parity mode's of few, uneven work items stay with
    64 heads a workgroup, lists that 16 heads cut nearly as finely or 64 heads take in one full round with those."""
    wide = lambda n, H, rows, precise, listed=False: attend_wide_items(n, H, rows, precise, listed) > 0
    for precise in (3, 4):
        for call in ((27, 128, 16384), (24, 112, 12000), (24, 128, 13000), (60, 64, 12000), (9, 256, 32768), (6, 384, 16384), (5, 384, 24000),
                     (7, 512, 24000), (1, 640, 32768), (3, 640, 24000), (3, 768, 24000), (3, 1024, 24000)):
            assert not wide(*call, precise), (call, precise)
        for call in ((17, 64, 9000), (18, 64, 10262), (12, 128, 6000), (18, 128, 9000), (17, 128, 13000), (9, 160, 6000), (3, 192, 24000),
                     (7, 256, 3000), (3, 384, 6000), (2, 768, 6000)):
            assert wide(*call, precise), (call, precise)
    for precise in (1, 2):
        assert not wide(3, 640, 16384, precise) and wide(2, 768, 24000, precise) and wide(17, 160, 24000, precise) and wide(5, 512, 12000, precise)
        assert not wide(64, 64, 2048, precise, True) and wide(16, 128, 4096, precise, True) and wide(48, 64, 2048, precise, True)
        assert not wide(3, 128, 8192, precise, True) and not wide(12, 80, 4096, precise, True) and wide(12, 160, 2048, precise, True)
    assert wide(3, 640, 16384, 0) and wide(64, 64, 2048, 0, True) and wide(3, 128, 8192, 0, True)
    assert not wide(3, 640, 8192, 4, True) and wide(3, 768, 2048, 4, True)
