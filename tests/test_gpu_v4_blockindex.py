"""The second cache format's block indexer on the device against the CPU oracle and against
the reference's own kernels, bit for bit: the Hadamard + fp4 spread and the block scorer."""
import numpy as np
import pytest

from rivoli_amd import hip
from tests.gpu_util import back, dev, dzeros, need_ref
from tests.test_gpu_v4 import same_bits
from tests.test_oracle_v4_blockindex import bf16_round

pytestmark = pytest.mark.gpu


def device_spread(x: np.ndarray, launch=None) -> np.ndarray:
    rows, d = x.shape
    buf = dev(x)
    if launch is None:
        hip.launch_act_quant_f4_rotated(buf, rows, d)
    else:
        assert launch(buf.data_ptr(), rows, d, None) == 0
    return back(buf, np.float32).reshape(x.shape)


def spread_rows(rows, d, seed):
    """bf16-valued rows (the reference's input dtype) over a wide range of magnitudes, with the
    special blocks: all zero, negative zero, below the amax floor, one outlier per block."""
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((rows, d)) * np.exp(rng.uniform(-6, 6, (rows, 1)))).astype(np.float32)
    if rows > 8:
        x[1] = 0.0
        x[2] = np.float32(-0.0)
        x[3] = np.float32(1e-38)
        x[4, ::32] *= np.float32(300.0)
        x[5] = np.float32(3.0)         # a constant row: one spike after the rotation
        x[6] = rng.standard_normal(d).astype(np.float32) * np.float32(1e-40)   # denormals: below the amax floor
        x[7] = rng.standard_normal(d).astype(np.float32) * np.float32(1e30)    # sums stay finite
    return bf16_round(x)


@pytest.mark.parametrize("rows,d", [(1, 128), (9, 128), (60, 128), (1000, 128), (7, 32), (33, 64), (129, 256),
                                    (4097, 128)])
def test_spread_matches_the_oracle(oracle, rows, d):
    x = spread_rows(rows, d, rows * 1000 + d)
    code, want = oracle.act_quant_f4_rotated(x)
    assert code == 0
    got = device_spread(x)
    bad = same_bits(got, want)
    assert bad.size == 0, [(int(i) // d, int(i) % d, got.ravel()[i], want.ravel()[i]) for i in bad[:6]]


@pytest.mark.parametrize("rows,d", [(8192, 128), (8193, 128), (16385, 64)])
def test_spread_across_the_change_of_rows_in_flight(oracle, rows, d):
    """Up to 8192 rows of 128 (16 384 of 64) a wave has one row group in flight, past them four."""
    x = spread_rows(rows, d, rows)
    assert same_bits(device_spread(x), oracle.act_quant_f4_rotated(x)[1]).size == 0


def sixty_binades():
    rng = np.random.default_rng(60)
    base = bf16_round(rng.standard_normal((60, 128)).astype(np.float32))
    return bf16_round(base * (2.0 ** (np.arange(60) - 30))[:, None].astype(np.float32))


def test_spread_over_sixty_binades(oracle):
    """crates/engine/tests/kernel_v4_indexer.rs:246-277: row r scaled into binade r - 30, so the
    block scale lands on 60 powers of two."""
    x = sixty_binades()
    code, want = oracle.act_quant_f4_rotated(x)
    assert same_bits(device_spread(x), want).size == 0
    scales = {float(np.abs(r[r != 0]).min()) for r in want if (r != 0).any()}
    assert len(scales) >= 55


def test_reference_spread_agrees_with_the_oracle_and_this_library(oracle):
    """The reference's own kernel (blockindex.hip compiled for this GPU): the sixty binades
    against the oracle, other widths against this library."""
    ref = need_ref("rivoli_act_quant_f4_rotated")
    x = sixty_binades()
    want = oracle.act_quant_f4_rotated(x)[1]
    assert same_bits(device_spread(x, launch=ref.rivoli_act_quant_f4_rotated), want).size == 0
    for rows, d in ((333, 256), (77, 128), (19, 64), (11, 32)):
        wide = spread_rows(rows, d, 5)
        assert same_bits(device_spread(wide, launch=ref.rivoli_act_quant_f4_rotated),
                         device_spread(wide)).size == 0, (rows, d)


def test_spread_guards():
    """blockindex.hip:241-257; kernel_v4_indexer.rs:287-320."""
    buf = dzeros(512 * 4)
    lib = hip.lib()
    call = lambda rows, d: lib.rivoli_act_quant_f4_rotated(buf.data_ptr(), rows, d, None)
    assert call(1, 128) == 0
    assert call(0, 128) == 1001 and call(1, 0) == 1001
    assert call(1, 512) == 1002
    assert call(1, 96) == 1003
    assert call(1, 16) == 1004
    assert lib.rivoli_act_quant_f4_rotated(None, 1, 128, None) == 1001
    assert lib.rivoli_act_quant_f4_rotated(buf.data_ptr() + 4, 1, 128, None) == 1004


# ---- the block scorer -------------------------------------------------------------------------

def device_score(q, kv, w, launch=None) -> np.ndarray:
    s, heads, hd = q.shape
    n_comp = kv.shape[0]
    qd, kd, wd = dev(q), dev(kv), dev(w)
    out = dzeros(s * n_comp * 4, 0x5A)
    if launch is None:
        hip.launch_index_score_blocks(qd, kd, wd, out, s, n_comp, heads, hd)
    else:
        assert launch(qd.data_ptr(), kd.data_ptr(), wd.data_ptr(), out.data_ptr(), s, n_comp, heads, hd, None) == 0
    return back(out, np.float32).reshape(s, n_comp)


def score_case(s, n_comp, heads, hd, seed, spread=None):
    """Arbitrary f32 operands make every addition round, so a reordered or fused dot shows;
    spread operands (oracle-made) are what the engine feeds."""
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((s, heads, hd)).astype(np.float32)
    kv = rng.standard_normal((n_comp, hd)).astype(np.float32)
    if spread is not None:
        q = spread.act_quant_f4_rotated(bf16_round(q).reshape(-1, hd))[1].reshape(s, heads, hd)
        kv = spread.act_quant_f4_rotated(bf16_round(kv))[1]
    w = bf16_round((rng.standard_normal((s, heads)) * hd ** -0.5).astype(np.float32))  # signed
    return q, kv, w


@pytest.mark.parametrize("s,n_comp,heads,hd,spread", [
    (1, 1, 64, 128, False), (2, 300, 64, 128, False), (33, 70, 8, 128, True), (5, 513, 64, 128, True),
    (3, 5, 4, 32, False), (2, 130, 3, 64, True), (1, 257, 2, 256, False), (40, 64, 64, 128, False),
    (1, 200, 128, 128, False), (1, 70, 130, 128, False), (2, 65, 5, 128, True), (300, 520, 3, 128, False),
])
def test_score_matches_the_oracle(oracle, s, n_comp, heads, hd, spread):
    q, kv, w = score_case(s, n_comp, heads, hd, s * 31 + n_comp, oracle if spread else None)
    code, want = oracle.index_score_blocks(q, kv, w)
    assert code == 0
    got = device_score(q, kv, w)
    bad = same_bits(got, want)
    assert bad.size == 0, [(int(i) // n_comp, int(i) % n_comp, got.ravel()[i], want.ravel()[i]) for i in bad[:6]]
    assert np.count_nonzero(want) > 0 or n_comp * s < 4


@pytest.mark.parametrize("n_comp", [1, 16, 17, 31, 32, 33, 65, 8192, 8193, 8225])
@pytest.mark.parametrize("heads", [1, 15, 16, 17, 64])
def test_one_query_at_the_edges_of_its_tiles(oracle, n_comp, heads):
    """Workgroups of 32 blocks (64 past 8192), waves of 16 or 32 heads; where `mixed`, some blocks' rows are not spread
    rows, so exact and folded workgroups meet in one launch."""
    for mixed in (False, True):
        q, kv, w = score_case(1, n_comp, heads, 128, n_comp + heads, oracle)
        if mixed:
            kv[40::97] *= np.float32(1.2345678)
        assert same_bits(device_score(q, kv, w), oracle.index_score_blocks(q, kv, w)[1]).size == 0, mixed


def test_score_known_answer(oracle):
    """kernel_v4_indexer.rs:689-726 (f32 accumulation, one bf16 round: 1.125, not 1.0)."""
    heads, hd = 64, 128
    kv = np.zeros((1, hd), np.float32)
    kv[0, 0] = 1.0
    q = np.zeros((1, heads, hd), np.float32)
    q[0, :, 0] = 2.0 ** -9
    q[0, 0, 0] = 1.0
    got = device_score(q, kv, np.ones((1, heads), np.float32))
    assert got[0, 0] == np.float32(1.125)


def test_reference_scorer_agrees_with_the_oracle_and_this_library(oracle):
    """The reference's own kernel (blockindex.hip compiled for this GPU) on rounding-sensitive
    operands."""
    ref = need_ref("rivoli_index_score_blocks")
    for shape in [(4, 200, 64, 128), (3, 77, 5, 64)]:
        q, kv, w = score_case(*shape, seed=9)
        theirs = device_score(q, kv, w, launch=ref.rivoli_index_score_blocks)
        assert same_bits(theirs, oracle.index_score_blocks(q, kv, w)[1]).size == 0
        assert same_bits(theirs, device_score(q, kv, w)).size == 0


def test_score_guards():
    """blockindex.hip:264-275."""
    buf = dzeros(4096)
    p = buf.data_ptr()
    lib = hip.lib()
    assert lib.rivoli_index_score_blocks(p, p, p, p, 1, 1, 1, 8, None) == 0
    assert lib.rivoli_index_score_blocks(p, p, p, p, 0, 1, 1, 8, None) == 1001
    assert lib.rivoli_index_score_blocks(p, p, p, p, 1, 1, 0, 8, None) == 1001
    assert lib.rivoli_index_score_blocks(p, p, p, p, 1, 1, 1, 0, None) == 1001
    assert lib.rivoli_index_score_blocks(p, p, p, p, 1, 0, 1, 8, None) == 1005
    assert lib.rivoli_index_score_blocks(None, p, p, p, 1, 1, 1, 8, None) == 1001


def test_prefill_sized_scores_on_sampled_rows_and_the_selection_they_feed(oracle):
    """A prefill chunk's worth (256 queries x 2048 blocks x 64 heads x 128): the oracle checks
    sampled query rows; then the chain the engine runs (crates/engine/src/v4/blocksel.rs:218-248
    followed by select.rs:153-188) — spread q, score, select — against the oracle's chain."""
    s, n_comp, heads, hd, k = 256, 2048, 64, 128, 512
    rng = np.random.default_rng(2048)
    q_raw = bf16_round(rng.standard_normal((s * heads, hd)).astype(np.float32))
    kv = oracle.act_quant_f4_rotated(bf16_round(rng.standard_normal((n_comp, hd)).astype(np.float32)))[1]
    w = bf16_round((rng.standard_normal((s, heads)) * hd ** -0.5).astype(np.float32))
    qd, kd, wd = dev(q_raw), dev(kv), dev(w)
    hip.launch_act_quant_f4_rotated(qd, s * heads, hd)
    score = dzeros(s * n_comp * 4, 0x5A)
    hip.launch_index_score_blocks(qd, kd, wd, score, s, n_comp, heads, hd)
    got = back(score, np.float32).reshape(s, n_comp)
    q = back(qd, np.float32).reshape(s, heads, hd)
    for t in (0, 1, 100, 255):
        want_q = oracle.act_quant_f4_rotated(q_raw.reshape(s, heads, hd)[t])[1]
        assert same_bits(q[t], want_q).size == 0
        code, want = oracle.index_score_blocks(want_q[None], kv, w[t:t + 1])
        assert same_bits(got[t:t + 1], want).size == 0, t
    sel = dzeros(s * k * 4)
    hip.launch_index_select_blocks(score, s, n_comp, 4, k, False, 0, sel)   # decode rule: every row ranks all blocks
    got_sel = back(sel, np.int32).reshape(s, k)
    for t in (0, 100, 255):
        want_sel = oracle.v4_scored_rows(got[t:t + 1], 4, k, False, 0)
        np.testing.assert_array_equal(got_sel[t], want_sel[0])


@pytest.mark.parametrize("s,n_comp,heads,hd,ratio", [(700, 175, 4, 128, 4), (300, 300, 2, 128, 1), (520, 130, 3, 64, 4),
                                                     (64, 16, 8, 128, 4), (1030, 100, 2, 128, 4)])
def test_prefill_form_writes_every_legal_entry_and_skips_whole_groups(oracle, s, n_comp, heads, hd, ratio):
    """score[t][c] for c < (t + 1) / ratio equals the full kernel's bit for bit; a 64-block group
    with no legal block for row t keeps the buffer's fill; the selection built on it is the one
    built on the full matrix."""
    q, kv, w = score_case(s, n_comp, heads, hd, s + ratio)
    full = device_score(q, kv, w)
    qd, kd, wd = dev(q), dev(kv), dev(w)
    out = dzeros(s * n_comp * 4, 0x5A)
    hip.launch_index_score_blocks_prefill(qd, kd, wd, out, s, n_comp, heads, hd, ratio)
    got = back(out, np.float32).reshape(s, n_comp)
    fill = np.frombuffer(b"\x5a" * 4, np.uint32)[0]
    limit = np.minimum((np.arange(s) + 1) // ratio, n_comp)
    cols = np.arange(n_comp)
    legal = cols[None, :] < limit[:, None]
    group_live = (cols[None, :] // 64) * 64 < limit[:, None]
    assert np.array_equal(got.view(np.uint32)[legal], full.view(np.uint32)[legal])
    assert np.array_equal(got.view(np.uint32)[group_live], full.view(np.uint32)[group_live])
    assert (got.view(np.uint32)[~group_live] == fill).all()
    assert (~group_live).any() and legal.any()
    k = min(32, n_comp)
    sel_a, sel_b = dzeros(s * k * 4), dzeros(s * k * 4)
    hip.launch_index_select_blocks(out, s, n_comp, ratio, k, True, 0, sel_a)
    hip.launch_index_select_blocks(dev(full), s, n_comp, ratio, k, True, 0, sel_b)
    assert np.array_equal(back(sel_a, np.int32), back(sel_b, np.int32))
    assert hip.lib().rivoli_index_score_blocks_prefill(qd.data_ptr(), kd.data_ptr(), wd.data_ptr(), out.data_ptr(),
                                                       s, n_comp, heads, hd, 0, None) == 1001


def few_bit_rows(rng, rows, span):
    """+-{1, 1.5} times powers of two over exactly `span` + 1 binades, with zeros; every third row
    positive and mostly at its top binade, so that a sum comes near the largest the rule allows."""
    e = rng.integers(0, span + 1, (rows, 128))
    e[::3][rng.random((len(e[::3]), 128)) < 0.9] = span
    e[:, 0], e[:, 1] = 0, span
    x = rng.choice([-1.5, -1.0, 1.0, 1.5], (rows, 128)) * 2.0 ** (e - 7)
    x[::3] = np.abs(x[::3])
    x[:, 2:][rng.random((rows, 126)) < 0.1] = 0.0
    return x.astype(np.float32)


@pytest.mark.parametrize("s,n_comp,heads", [(1, 1, 64), (2, 65, 31), (4, 190, 17), (5, 33, 1), (9, 3100, 64), (16, 1600, 47),
                                            (23, 1210, 16)])
@pytest.mark.parametrize("q_span,kv_span", [(3, 4), (6, 7), (13, 0), (7, 7), (3, 20)])
def test_score_of_rows_whose_sums_are_exact_up_to_the_last_span_and_past_it(oracle, s, n_comp, heads, q_span, kv_span):
    """Rows of one- and two-bit values over q_span + kv_span = 7 and 13 binades, where every sum is
    exact and the matrix cores take them, and 14 and 23, where they are folded term by term; then
    the same launch with a single block, and a single head, that only the fold gets right. All bit
    for bit, through the few-query and the many-query kernel and both forms of the call."""
    rng = np.random.default_rng(s * 1000 + n_comp + q_span * 7 + kv_span)
    q = few_bit_rows(rng, s * heads, q_span).reshape(s, heads, 128)
    kv = few_bit_rows(rng, n_comp, kv_span)
    w = bf16_round((rng.standard_normal((s, heads)) * 0.1).astype(np.float32))
    for change in ("none", "block", "head"):
        if change == "block":
            kv[n_comp // 2] = rng.standard_normal(128).astype(np.float32)
        if change == "head":
            q[s // 2, heads // 2] = rng.standard_normal(128).astype(np.float32)
        code, want = oracle.index_score_blocks(q, kv, w)
        got = device_score(q, kv, w)
        assert code == 0 and same_bits(got, want).size == 0, change
        out = dzeros(s * n_comp * 4, 0x5A)
        hip.launch_index_score_blocks_prefill(dev(q), dev(kv), dev(w), out, s, n_comp, heads, 128, 1)
        part = back(out, np.float32).reshape(s, n_comp).view(np.uint32)
        live = (np.arange(n_comp)[None, :] // 64) * 64 < np.minimum(np.arange(s) + 1, n_comp)[:, None]
        assert np.array_equal(part[live], want.view(np.uint32)[live]) and (part[~live] == 0x5A5A5A5A).all(), change


@pytest.mark.parametrize("s,n_comp,heads,ratio", [(113, 300, 64, 0), (113, 300, 5, 4), (8185, 2100, 3, 0), (8185, 2100, 2, 4)])
def test_score_where_single_tiles_of_a_group_are_folded_and_past_64_tiles_of_a_split(oracle, s, n_comp, heads, ratio):
    """Blocks that only the fold gets right in the upper 32 of a group of 64, in the lower, in both and
    in none: a wave folds whole groups for its two queries and single tiles a half for each. 8 185
    queries by 2 100 blocks walk 66 tiles in one workgroup. Bit for bit on sampled queries."""
    rng = np.random.default_rng(s + n_comp + heads)
    q = few_bit_rows(rng, s * heads, 3).reshape(s, heads, 128)
    kv = few_bit_rows(rng, n_comp, 4)
    for c in (40, 64 + 3, 128 + 1, 160 + 1, 299, 2060, 2099):
        if c < n_comp:
            kv[c] = rng.standard_normal(128).astype(np.float32)
    w = bf16_round((rng.standard_normal((s, heads)) * 0.1).astype(np.float32))
    out = dzeros(s * n_comp * 4, 0x5A)
    if ratio:
        hip.launch_index_score_blocks_prefill(dev(q), dev(kv), dev(w), out, s, n_comp, heads, 128, ratio)
    else:
        hip.launch_index_score_blocks(dev(q), dev(kv), dev(w), out, s, n_comp, heads, 128)
    got = back(out, np.uint32).reshape(s, n_comp)
    for t in (0, 1, 7, 8, s // 2, s // 2 + 1, s - 2, s - 1):
        code, want = oracle.index_score_blocks(q[t:t + 1], kv, w[t:t + 1])
        live = (np.arange(n_comp) // 64) * 64 < (min((t + 1) // ratio, n_comp) if ratio else n_comp)
        assert code == 0 and np.array_equal(got[t][live], want[0].view(np.uint32)[live]), t
        assert (got[t][~live] == 0x5A5A5A5A).all(), t


@pytest.mark.parametrize("s,n_comp", [(1, 70), (9, 3100)])
@pytest.mark.parametrize("exponent", [59, 60, -59, -60])
def test_score_at_the_largest_and_smallest_exponents_whose_sums_are_exact(oracle, s, n_comp, exponent):
    """112 products of 2.25 * 2^120, two more and then fourteen of the other sign: a fold passes the
    largest float at the 114th and stays infinite, a sum in another order never reaches it. Rows of
    exponent 60 have to be folded; at 59 (and at -59, below which products leave the normal
    numbers' exact range) every order agrees."""
    q = np.full((s, 16, 128), 1.5 * 2.0 ** exponent, np.float32)
    kv = q[0, :1].repeat(n_comp, 0)
    q[:, :, 114:] *= np.float32(-1.0)
    w = np.full((s, 16), 0.25, np.float32)
    code, want = oracle.index_score_blocks(q, kv, w)
    assert code == 0 and np.isinf(want).all() == (exponent == 60)
    assert same_bits(device_score(q, kv, w), want).size == 0


def coded_rows(rng, rows, exponents):
    """Rows of e2m1 codes, each block of 32 times 2 to its exponent (`exponents` [rows][4]) and with a 4 or a 6."""
    x = rng.choice(np.array([0.0, -0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]), (rows, 4, 32)) * rng.choice([-1.0, 1.0], (rows, 4, 32))
    x[:, :, 5] = rng.choice([4.0, 6.0], (rows, 4))
    return (x * 2.0 ** np.asarray(exponents, np.float64)[:, :, None]).reshape(rows, 128).astype(np.float32)


@pytest.mark.parametrize("s,n_comp,heads", [(2060, 230, 64), (2060, 161, 49), (2060, 193, 33), (1380, 390, 64)])
def test_score_at_the_edges_of_what_the_fp4_products_take(oracle, s, n_comp, heads):
    """Each wave's two queries are of one kind: at and just past every bound under which dots come from the block-scaled fp4
    instruction, clamped and scaled (block exponents 9 apart, heads 20 binades, weights 2^+-50, scores scaled back by
    2^-20 and 2^40), rows of zeros and values that are no code. The blocks' rows likewise, in tiles of their own.
    Bit for bit on three waves of each kind, in both forms."""
    rng = np.random.default_rng(s + n_comp + heads)
    def at(e):  # every row's exponents
        return np.broadcast_to(np.asarray(e), (2 * heads, 4))
    def one_head(e, other):  # one head apart from the others
        x = np.full((2 * heads, 4), e)
        x[heads // 2] = other
        return x
    kinds = [at([0, 0, 1, 0]), at([5, 0, 3, 1]), at([6, 0, 3, 1]), one_head(0, -20), one_head(0, -21), at([0, 0, 0, 0]), at([0, 0, 0, 0]),
             at([30, 30, 30, 29]), at([31, 30, 30, 30]), at([-29, -29, -29, -29]), at([-30, -30, -30, -30]), at([0, 0, 0, 0]), at([1, 0, 0, 0]),
             at([1, 0, 0, 0]), at([0, 1, 0, 0])]
    q = np.zeros((s, heads, 128), np.float32)
    w = bf16_round((rng.standard_normal((s, heads)) * 0.1).astype(np.float32))
    for pair in range(s // 2):
        k = pair % len(kinds)
        rows = coded_rows(rng, 2 * heads, kinds[k])
        if k == 11: rows[:] = 0.0
        if k == 12: rows[::3, 32:64] = 0.0
        if k == 13: rows[heads - 1, 7] = 0.75          # half of a code's smallest step
        if k == 14: rows[1] = rng.standard_normal(128)
        q[2 * pair:2 * pair + 2] = rows.reshape(2, heads, 128)
        if k == 5: w[2 * pair, ::2], w[2 * pair + 1, 1::3] = 2.0 ** 50, 1.5 * 2.0 ** -50
        if k == 6: w[2 * pair, 0], w[2 * pair + 1, 1] = 2.0 ** 51, 1.5 * 2.0 ** -51
    kv = coded_rows(rng, n_comp, np.where(np.arange(n_comp)[:, None] // 64 == 1, [0, 4, 1, 0], [0, 0, -1, 0]))
    kv[70] = 0.0
    kv[75, 96:] = 0.0
    kv[n_comp - 1] = rng.standard_normal(128)
    kv[n_comp - 2, 3] = 0.25
    # (the scores' scale with exponents e and f: e + f + 13; the first blocks' f is 0, 64 to 127's is 4)
    pairs = [len(kinds) * r + k for r in (0, 40, (s // 2 - len(kinds)) // len(kinds)) for k in range(len(kinds))]
    queries = np.array([2 * p + i for p in pairs for i in (0, 1)] + [s - 1])
    code, want = oracle.index_score_blocks(q[queries], kv, w[queries])
    assert code == 0 and np.isfinite(want).all()
    qd, kd, wd = dev(q), dev(kv), dev(w)
    for ratio in (0, 4):
        out = dzeros(s * n_comp * 4, 0x5A)
        if ratio:
            hip.launch_index_score_blocks_prefill(qd, kd, wd, out, s, n_comp, heads, 128, ratio)
        else:
            hip.launch_index_score_blocks(qd, kd, wd, out, s, n_comp, heads, 128)
        got = back(out, np.uint32).reshape(s, n_comp)[queries]
        live = np.ones(got.shape, bool) if not ratio else \
            (np.arange(n_comp)[None, :] // 64) * 64 < np.minimum((queries + 1) // ratio, n_comp)[:, None]
        bad = np.argwhere((got != want.view(np.uint32)) & live)
        assert bad.size == 0, (ratio, [(int(queries[i]), int(queries[i]) // 2 % len(kinds), int(c)) for i, c in bad[:6]])
        assert (got[~live] == 0x5A5A5A5A).all()


def check_scores(q, kv, w, queries, want, what):
    """Both forms of a launch of q [s][heads][128] against the oracle's scores of some of its queries, bit for bit; entries that the
    prefill form has no use for stay as they were."""
    s, heads = w.shape
    n_comp = len(kv)
    qd, kd, wd = dev(q), dev(kv), dev(w)
    for ratio in (0, 4):
        out = dzeros(s * n_comp * 4, 0x5A)
        if ratio:
            hip.launch_index_score_blocks_prefill(qd, kd, wd, out, s, n_comp, heads, 128, ratio)
        else:
            hip.launch_index_score_blocks(qd, kd, wd, out, s, n_comp, heads, 128)
        got = back(out, np.uint32).reshape(s, n_comp)[queries]
        live = np.ones(got.shape, bool) if not ratio else \
            (np.arange(n_comp)[None, :] // 64) * 64 < np.minimum((queries + 1) // ratio, n_comp)[:, None]
        bad = np.argwhere((got != want.view(np.uint32)) & live)
        assert bad.size == 0, (what, ratio, len(bad), [(int(queries[i]), int(c)) for i, c in bad[:6]])
        assert (got[~live] == 0x5A5A5A5A).all()


@pytest.mark.parametrize("s,n_comp,heads", [(2060, 230, 64), (2060, 201, 33), (1380, 390, 64)])
def test_score_of_rows_with_the_smallest_codes(oracle, s, n_comp, heads):
    """Blocks of 0 and +-2^-127, which are half a code under the smallest normal scale and are no zeros, in rows with larger blocks and in rows
    of nothing else; blocks whose largest value is 2^-126 to 2^-124; and spread rows of such amplitude, which is below the spread's
    floor. Of q in waves of their own, of kv in tiles of their own."""
    rng = np.random.default_rng(s + n_comp + heads)
    least = np.float32(2.0 ** -127)

    def spread(rows, amplitude):
        x = bf16_round((rng.standard_normal((rows, 128)) * amplitude).astype(np.float32))
        code, x = oracle.act_quant_f4_rotated(x)
        assert code == 0 and (x != 0).any()
        return x

    def tiny(rows, kind):
        if kind >= 6:
            x = spread(rows, (0.12, 0.3, 1.0)[kind - 6] * 2.0 ** -126)
            assert kind > 6 or np.abs(x).max() == least
            return x
        if kind >= 2:  # the largest value 4 or 6 times 2^-128 to 2^-125
            return coded_rows(rng, rows, np.full((rows, 4), (-128, -127, -126, -125)[kind - 2]))
        x = coded_rows(rng, rows, np.zeros((rows, 4)))
        small = rng.choice(np.array([0.0, -0.0, least, -least], np.float32), (rows, 128))
        small[:, 5::32] = least
        if kind == 1:
            return small
        x[:, 32:64] = small[:, 32:64]
        return x

    q = np.zeros((s, heads, 128), np.float32)
    w = bf16_round((rng.standard_normal((s, heads)) * 0.1).astype(np.float32))
    rows_of = [[tiny(2 * heads, kind) if kind >= 0 else spread(2 * heads, 1.0) * np.float32(2.0 ** 20) for _ in range(6)] for kind in range(-2, 9)]
    for pair in range(s // 2):  # (two of eleven waves with rows as usual)
        q[2 * pair:2 * pair + 2] = rows_of[pair % 11][pair // 11 % 6].reshape(2, heads, 128)
    kv = spread(n_comp, 1.0)
    for kind in range(6):  # a row of each in tiles that would be taken otherwise, and whole ones
        at = 32 * kind + 7
        if at + 2 < n_comp:
            kv[at:at + 2] = tiny(2, kind)
    kv[-5:] = tiny(5, 6)
    pairs = [11 * r + k for r in (0, 30, (s // 2 - 11) // 11) for k in range(11)]
    queries = np.array([2 * p + i for p in pairs for i in (0, 1)])
    code, want = oracle.index_score_blocks(q[queries], kv, w[queries])
    assert code == 0 and np.isfinite(want).all()
    check_scores(q, kv, w, queries, want, "smallest codes")
    # the rest of the blocks as usual: only q has such rows
    kv = spread(n_comp, 1.0)
    code, want = oracle.index_score_blocks(q[queries], kv, w[queries])
    check_scores(q, kv, w, queries, want, "smallest codes of q")
    # and the other way round
    q[:] = np.repeat(spread(2 * heads, 1.0), -(-s // 2), axis=0)[:s * heads].reshape(s, heads, 128)
    kv[40:44] = tiny(4, 0)
    kv[70:74] = tiny(4, 1)
    kv[100:164] = tiny(64, 1)
    kv[n_comp - 9:] = tiny(9, 6)
    code, want = oracle.index_score_blocks(q[queries], kv, w[queries])
    check_scores(q, kv, w, queries, want, "smallest codes of kv")


@pytest.mark.parametrize("s,n_comp,heads", [(2060, 230, 64), (2060, 201, 33)])
def test_score_keeps_the_last_bit_of_the_largest_sums_that_the_fp4_products_take(oracle, s, n_comp, heads):
    """Block exponents that span 9 over both rows, three blocks at the top and one at the bottom, that one in each half of the products'
    contraction. One-signed sums of the top blocks come to the middle between two bf16 numbers, cancelling ones to zero: the
    bottom block's sum, down to the last unit, decides. One head a query has a weight, so that its dot is the score."""
    rng = np.random.default_rng(s + heads)
    n_kinds = 16  # the bottom block, whether the top blocks cancel, and 9 binades in q alone or 5 in q and 4 in kv
    q = np.zeros((s, heads, 128), np.float32)
    w = np.zeros((s, heads), np.float32)
    w[np.arange(s), np.arange(s) // 2 % heads] = 1.0
    for pair in range(s // 2):
        low, cancel, apart = pair % 4, pair // 4 % 2, (9, 5)[pair // 8 % 2]
        rows = np.empty((2 * heads, 128), np.float32)
        for r in rows if pair < 5 * n_kinds else ():
            # a sum of 4 x 96 + 2 x sixes, times a block's 4 or 6: a middle for sixes odd, or two more than a multiple of four
            sixes = int(rng.choice(np.arange(65, 96, 2))) if rng.random() < 0.5 else int(rng.choice(np.arange(66, 96, 4)))
            top = rng.permutation(np.where(np.arange(96) < sixes, 6.0, 4.0))
            if cancel:
                top = rng.permutation(np.concatenate([top[:48], -top[:48]]))
            bottom = rng.choice([0.5, -0.5], 32)
            bottom[rng.integers(32)] = rng.choice([4.0, -4.0])
            values = np.insert(top, 32 * low, bottom * 2.0 ** -apart)
            r[:] = values * (1.0 if cancel else rng.choice([1.0, 1.0, -1.0]))
        q[2 * pair:2 * pair + 2] = rows.reshape(2, heads, 128) if pair < 5 * n_kinds else q[2 * pair - 10 * n_kinds:][:2]
    kv = np.repeat(rng.choice(np.array([6.0, 4.0], np.float32), n_comp)[:, None], 128, axis=1)
    for c in range(64, 128):  # of which a block is four binades down, with the smallest code in it, for the rows of 5
        b = c % 4
        kv[c, 32 * b:32 * b + 32] *= np.float32(2.0 ** -4)
        kv[c, 32 * b + 1:32 * b + 9] = np.float32(0.5 * 2.0 ** -4)
    pairs = [n_kinds * r + k for r in (0, 25, s // 2 // n_kinds - 1) for k in range(n_kinds)]
    queries = np.array([2 * p + i for p in pairs for i in (0, 1)])
    code, want = oracle.index_score_blocks(q[queries], kv, w[queries])
    # the dots by themselves, and without the bottom blocks: it is these that decide
    dots = np.einsum("thd,cd,th->tc", q[queries].astype(np.float64), kv.astype(np.float64), w[queries].astype(np.float64))
    top_q = np.where(np.abs(q[queries]) >= 4, q[queries], 0).astype(np.float64)
    top = np.einsum("thd,cd,th->tc", top_q, kv.astype(np.float64), w[queries].astype(np.float64))
    taken = np.full(want.shape, True)
    taken[:, 64:128] = (queries // 2 // 8 % 2 == 1)[:, None]
    assert code == 0 and np.array_equal(want[taken], np.maximum(bf16_round(dots.astype(np.float32)), 0)[taken])
    assert (bf16_round(dots.astype(np.float32)) != bf16_round(top.astype(np.float32)))[taken].mean() > 0.3
    check_scores(q, kv, w, queries, want, "the largest sums")
