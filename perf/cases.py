"""The work a program has this library do, as cases that can be timed and compared.

Every case is one pass of one layer through the `launch_*` entry points of `rivoli_amd.hip`, at a
size of the benchmark's or the tests' own workloads or between them: decode, prefill, sparse
selection and attention over the paged fp8 cache, and the same four over the second cache
format. `listed()` names the ones quoted; `draw()` makes more of the same ranges.

Buffers that a serving program owns for the life of a layer (pools, block tables, workspaces,
score and output buffers, compressor state) are made by `prepare`; `run` launches only.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rivoli_amd import hip

W, PT = 576, 64                      # latent 512 + rope 64; tokens per page
KVL, ROPE = 512, 64
ROW, REC = 2 * W, W + 4              # a bf16 row; a stored record (codes + one f32 scale)
INDEX_HEADS, INDEX_DIM = 64, 128
V4_DIM, V4_QUANT, V4_BLOCK = 512, 448, 64
V4_WINDOW, V4_RATIO, V4_CAP, V4_HEADS = 128, 4, 512, 64
V4_EPS = 1e-6


def listed():
    return [
        # one user's next token at a short context: append one row, gather 4096 (configuration 1)
        dict(name="decode_b1_4k", kind="decode", batch=1, ctx=4096, ragged=False, lens=1),
        # a full decode batch with contexts spread over 1024..32768 (configuration 3 as written)
        dict(name="decode_b32_ragged", kind="decode", batch=32, ctx=32768, ragged=True, lens=3),
        # a prompt's rows quantized into the cache (configuration 2)
        dict(name="append_8192", kind="append", tokens=8192),
        # sparse decode over long contexts, rows handed on as bf16 (configuration 4)
        dict(name="dsa_gather_b16_64k", kind="dsa_gather", batch=16, ctx=65536, k=2048),
        # sparse decode at 16k: keys appended, scored, 2048 rows selected and attended
        dict(name="dsa_attend_b8_16k", kind="dsa_attend", batch=8, ctx=16384, k=2048, heads=64, precise=2, lens=5),
        # dense decode attention at the metric point, 8-bit matrix instructions
        dict(name="attend_b32_32k", kind="attend", batch=32, ctx=32768, heads=64, precise=4, ragged=False, lens=6),
        # a small ragged batch in the parity mode
        dict(name="attend_b6_ragged", kind="attend", batch=6, ctx=9000, heads=64, precise=2, ragged=True, lens=7),
        # one token of the single-sequence engine over its linear slabs, reference signatures
        dict(name="engine_token_8k", kind="engine", nt=8192, k=2048, heads=64),
        # second format, a prompt of odd length: cache rows and pooled rows
        dict(name="v4_cache_8191", kind="v4_cache", tokens=8191, ratio=4),
        # second format, a prompt's block scores and selection
        dict(name="v4_index_8192", kind="v4_index", tokens=8192),
        # second format, a prompt's attention over [window | selected blocks]
        dict(name="v4_attend_8192", kind="v4_attend", tokens=8192),
        # second format, one token at 32k of context, on a position that closes a block
        dict(name="v4_decode_32k", kind="v4_decode", pos=32767),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm (odd ones as likely as even)."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "append", "dsa_gather", "dsa_attend", "attend", "attend", "engine",
                       "v4_cache", "v4_index", "v4_attend", "v4_decode"])
    lens = rng.randrange(1, 1 << 20)
    if kind == "decode":
        return dict(kind=kind, batch=_log(rng, 1, 32), ctx=_log(rng, 256, 16384), ragged=rng.random() < 0.7, lens=lens)
    if kind == "append":
        return dict(kind=kind, tokens=_log(rng, 64, 65536))
    if kind == "dsa_gather":
        return dict(kind=kind, batch=_log(rng, 1, 16), ctx=_log(rng, 3000, 65536), k=rng.choice([512, 1024, 2048]))
    if kind == "dsa_attend":
        return dict(kind=kind, batch=_log(rng, 1, 16), ctx=_log(rng, 3000, 65536), k=rng.choice([512, 1024, 2048]),
                    heads=rng.choice([16, 64, 64, 128]), precise=rng.choice([2, 4]), lens=lens)
    if kind == "attend":
        return dict(kind=kind, batch=_log(rng, 1, 32), ctx=_log(rng, 300, 16384), heads=rng.choice([16, 64, 64, 128]),
                    precise=rng.choice([0, 2, 2, 4]), ragged=rng.random() < 0.7, lens=lens)
    if kind == "engine":
        nt = _log(rng, 2100, 65536)
        return dict(kind=kind, nt=nt, k=rng.choice([512, 1024, 2048]), heads=64)
    if kind == "v4_cache":
        return dict(kind=kind, tokens=_log(rng, 300, 8192), ratio=rng.choice([4, 4, 128]))
    if kind in ("v4_index", "v4_attend"):
        return dict(kind=kind, tokens=_log(rng, 300, 8000))
    return dict(kind=kind, pos=_log(rng, 600, 65535))


# ---- sizes ---------------------------------------------------------------------------------

def _lens(case):
    """Context lengths, part of the case and not of the seed: uniform in [ctx / 32, ctx] or all ctx."""
    b, ctx = case["batch"], case["ctx"]
    if not case.get("ragged", True):
        return np.full(b, ctx, np.int32)
    lo = max(1, ctx // 32)
    if case["kind"] == "dsa_attend":     # contexts long enough to be worth a selection
        lo = max(ctx // 2, min(ctx, case["k"] + 1))
    return np.random.default_rng(case["lens"]).integers(lo, ctx + 1, size=b).astype(np.int32)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        lens = _lens(case)
        n = int(lens.sum())
        return dict(bytes=n * (REC + ROW) + int((-(-lens // PT)).sum()) * 4 + case["batch"] * (ROW + 4 + REC), flops=0)
    if kind == "append":
        return dict(bytes=case["tokens"] * (ROW + 4 + REC), flops=0)
    if kind == "dsa_gather":
        b, nt, k = case["batch"], case["ctx"], min(case["k"], case["ctx"])
        return dict(bytes=b * (nt * 4 + -(-nt // PT) * 4 + k * (4 + REC + ROW)), flops=0)
    if kind == "dsa_attend":
        lens, h = _lens(case), case["heads"]
        n, k, b = int(lens.sum()), int(np.minimum(lens, case["k"]).sum()), case["batch"]
        return dict(bytes=n * (INDEX_DIM * 2 + 4) + k * (4 + REC) + b * (INDEX_HEADS * (INDEX_DIM + 1) * 4 +
                                                                         h * (W + KVL) * 4),
                    flops=n * INDEX_HEADS * INDEX_DIM * 2 + k * h * 2 * (W + KVL))
    if kind == "attend":
        n, h = int(_lens(case).sum()), case["heads"]
        return dict(bytes=n * REC + case["batch"] * h * (W + KVL) * 4, flops=n * h * 2 * (W + KVL))
    if kind == "engine":
        nt, k, h = case["nt"], min(case["k"], case["nt"]), case["heads"]
        return dict(bytes=nt * (INDEX_DIM * 2 + 4) + k * (4 + KVL + 16 + 2 * ROPE) + h * (W + KVL) * 4 +
                    INDEX_HEADS * INDEX_DIM * 4, flops=nt * INDEX_HEADS * INDEX_DIM * 2 + k * h * 2 * (W + KVL))
    if kind == "v4_cache":
        n, ratio = case["tokens"], case["ratio"]
        cd = V4_DIM * (2 if ratio == 4 else 1)
        return dict(bytes=n * V4_QUANT * 8 + 2 * n * cd * 4 + (n // ratio) * V4_DIM * 4, flops=0)
    if kind == "v4_index":
        n = case["tokens"]
        n_comp = n // V4_RATIO
        legal = int(np.minimum((np.arange(n) + 1) // V4_RATIO, n_comp).sum())
        return dict(bytes=n * INDEX_HEADS * (INDEX_DIM * 8 + 4) + n_comp * INDEX_DIM * 4 + legal * 4 +
                    n * (min(n, V4_WINDOW) + min(V4_CAP, n_comp)) * 4, flops=legal * INDEX_HEADS * INDEX_DIM * 2)
    if kind == "v4_attend":
        n = case["tokens"]
        n_comp = n // V4_RATIO
        cap = min(V4_CAP, n_comp)
        t = np.arange(n) + 1
        live = int(np.minimum(t, V4_WINDOW).sum() + np.minimum(t // V4_RATIO, cap).sum())
        return dict(bytes=n * V4_HEADS * V4_DIM * 8 + (n + n_comp) * V4_DIM * 4 + n * (min(n, V4_WINDOW) + cap) * 4,
                    flops=live * V4_HEADS * V4_DIM * 4)
    n_comp = (case["pos"] + 1) // V4_RATIO
    slots = V4_WINDOW + min(V4_CAP, n_comp)
    return dict(bytes=n_comp * (INDEX_DIM + 1) * 4 + slots * V4_DIM * 4 + V4_HEADS * V4_DIM * 8 +
                INDEX_HEADS * INDEX_DIM * 8 + 16 * V4_DIM * 4 + 16 * INDEX_DIM * 4,
                flops=n_comp * INDEX_HEADS * INDEX_DIM * 2 + slots * V4_HEADS * V4_DIM * 4)


def tolerance(case):
    kind = case["kind"]
    if kind in ("decode", "append", "dsa_gather", "v4_index"):
        return "exact"                      # stored bytes, selections, one correctly rounded product
    if kind == "engine":                    # against float64 3e-6 (worst element 1.6e-5)
        return dict(rel=2e-5, max=2e-4)
    if kind in ("dsa_attend", "attend"):
        # against float64, on caches with outlier rows: q and the softmax weights as bf16 hi + lo
        # 1.3e-5 (worst element 4e-4), as three and two e4m3 terms 1.4e-4 (6e-3), once bf16 1.1e-2
        return {2: dict(rel=5e-5, max=2e-3), 4: dict(rel=6e-4, max=0.025), 0: dict(rel=0.03, max=1.0)}[case["precise"]]
    if kind == "v4_cache":
        # a pooled value one bf16 rounding off may land on the next 8-bit step (1/8 of it), and a block's
        # largest may move its power-of-two scale; float64 pooling in the same steps differs by 1e-2
        return dict(rel=5e-3, max=0.3)
    # against float64 9e-4 to 1e-3 (worst element 4e-3): outputs rounded to bf16
    return dict(rel=4e-3, max=0.05)


# ---- inputs --------------------------------------------------------------------------------

class _Maker:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda", dtype=torch.float32)

    def rows(self, n, width, share, gain):
        """Rows ~N(0, 1), `share` of them `gain` times larger (the outlier tokens of real caches)."""
        x = self.normal(n, width)
        x[self.uniform(n) < share] *= gain
        return x

    def tables(self, batch, blocks):
        """Block tables over a shuffled pool."""
        return torch.randperm(batch * blocks, generator=self.g, device="cuda").to(torch.int32).reshape(batch, blocks)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _zeros(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype, device="cuda")


def _slots(tables, seq, pos):
    """Cache slots of positions `pos` of sequences `seq`."""
    return tables[seq, pos // PT] * PT + (pos % PT).to(torch.int32)


def _filled_pool(mk, tables, lens):
    """A latent cache holding `lens` tokens per sequence."""
    n_pages = tables.numel()
    pool = _zeros(n_pages * hip.kv_page_bytes(PT, W), dtype=torch.uint8)
    seq = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), torch.from_numpy(lens.astype(np.int64)).cuda())
    pos = torch.cat([torch.arange(int(n), device="cuda") for n in lens])
    slots = _slots(tables, seq, pos).contiguous()
    for a in range(0, len(pos), 1 << 18):
        rows = mk.rows(min(1 << 18, len(pos) - a), W, 0.005, 50.0).bfloat16()
        hip.launch_kv_append_paged(rows, slots[a:], pool, len(rows), W, PT, n_pages)
    return pool, slots


def _next_slots(tables, lens):
    last = torch.from_numpy(lens.astype(np.int64) - 1).cuda()
    return _slots(tables, torch.arange(len(lens), device="cuda"), last).contiguous()


def prepare(case, seed):
    mk = _Maker(seed)
    st = dict(globals()["_prepare_" + case["kind"]](case, mk), kind=case["kind"])
    torch.cuda.synchronize()
    return st


def run(st):
    return globals()["_run_" + st["kind"]](st, torch.cuda.current_stream().cuda_stream)


# ---- fp8 paged cache: append and gather ----------------------------------------------------

def _prepare_decode(case, mk):
    lens = _lens(case)
    b, blocks = case["batch"], -(-case["ctx"] // PT)
    tables = mk.tables(b, blocks)
    pool, _ = _filled_pool(mk, tables, lens)
    cu = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
    return dict(pool=pool, tables=tables, lens=torch.from_numpy(lens).cuda(), cu=cu, b=b, blocks=blocks,
                total=int(lens.sum()), n_pages=b * blocks, slots=_next_slots(tables, lens),
                new=mk.normal(b, W).bfloat16(), out=_empty(int(lens.sum()), W, dtype=torch.bfloat16))


def _run_decode(st, s):
    hip.launch_kv_append_paged(st["new"], st["slots"], st["pool"], st["b"], W, PT, st["n_pages"], None, s)
    hip.launch_kv_gather_paged_packed(st["pool"], st["tables"], st["lens"], st["cu"], st["out"], st["b"], st["blocks"],
                                      st["total"], W, PT, st["n_pages"], None, s)
    return st["out"]


def _prepare_append(case, mk):
    n = case["tokens"]
    tables = mk.tables(1, -(-n // PT))
    pos = torch.arange(n, device="cuda")
    return dict(n=n, n_pages=tables.numel(), rows=mk.rows(n, W, 0.005, 50.0).bfloat16(),
                slots=_slots(tables, torch.zeros_like(pos), pos).contiguous(),
                pool=_zeros(tables.numel() * hip.kv_page_bytes(PT, W), dtype=torch.uint8))


def _run_append(st, s):
    hip.launch_kv_append_paged(st["rows"], st["slots"], st["pool"], st["n"], W, PT, st["n_pages"], None, s)
    return st["pool"]


# ---- sparse selection ----------------------------------------------------------------------

def _prepare_dsa_gather(case, mk):
    b, nt, k = case["batch"], case["ctx"], case["k"]
    blocks = -(-nt // PT)
    tables = mk.tables(b, blocks)
    pool, _ = _filled_pool(mk, tables, np.full(b, nt, np.int32))
    scores = mk.normal(b, nt)
    scores[:, -64:] += 4.0                       # the recency boost
    return dict(b=b, nt=nt, k=k, blocks=blocks, tables=tables, pool=pool, n_pages=b * blocks, scores=scores,
                ws=_zeros(max(hip.index_topk_workspace_bytes(b, nt), 16), dtype=torch.uint8),
                rows=_zeros(b, k, dtype=torch.int32), out=_zeros(b, k, W, dtype=torch.bfloat16))


def _run_dsa_gather(st, s):
    hip.launch_dsa_select_gather_paged(st["scores"], st["b"], st["nt"], None, st["nt"], st["k"], st["rows"], st["ws"],
                                       False, st["pool"], st["tables"], st["out"], st["blocks"], W, PT, st["n_pages"],
                                       None, s)
    return st["rows"], st["out"]


def _prepare_dsa_attend(case, mk):
    lens = _lens(case)
    b, k, h = case["batch"], case["k"], case["heads"]
    nt, blocks = int(lens.max()), -(-case["ctx"] // PT)
    tables = mk.tables(b, blocks)
    pool, slots = _filled_pool(mk, tables, lens)
    kpool = _zeros(b * blocks * PT, INDEX_DIM, dtype=torch.bfloat16)
    hip.launch_index_append_paged(mk.normal(len(slots), INDEX_DIM), slots, kpool, len(slots), INDEX_DIM, PT, b * blocks)
    return dict(b=b, k=k, h=h, nt=nt, blocks=blocks, tables=tables, pool=pool, n_pages=b * blocks, kpool=kpool,
                precise=case["precise"], lens=torch.from_numpy(lens).cuda(), slots=_next_slots(tables, lens),
                key=mk.normal(b, INDEX_DIM), iq=mk.normal(b, INDEX_HEADS, INDEX_DIM), iw=mk.uniform(b, INDEX_HEADS),
                scores=_zeros(b, nt), ws=_zeros(max(hip.index_topk_workspace_bytes(b, nt), 16), dtype=torch.uint8),
                rows=_zeros(b, k, dtype=torch.int32), n_rows=torch.from_numpy(np.minimum(lens, k).astype(np.int32)).cuda(),
                qabs=mk.normal(b, h, KVL), qrope=mk.normal(b, h, ROPE), clat=_empty(b, h, KVL),
                partial=_empty(max(hip.mla_attend_paged_scratch_floats(b, h, k), 4)))


def _run_dsa_attend(st, s):
    b, nt, k, n_pages = st["b"], st["nt"], st["k"], st["n_pages"]
    hip.launch_index_append_paged(st["key"], st["slots"], st["kpool"], b, INDEX_DIM, PT, n_pages, None, s)
    hip.launch_index_score_paged(st["iq"], st["iw"], st["kpool"], st["tables"], st["lens"], None, b, st["blocks"], nt,
                                 nt, INDEX_HEADS, INDEX_HEADS, INDEX_DIM, PT, n_pages, INDEX_DIM ** -0.5, 1.0,
                                 st["scores"], s)
    hip.launch_index_topk_batched(st["scores"], b, nt, st["lens"], nt, k, st["rows"], st["ws"], s)
    hip.launch_mla_attend_paged(st["qabs"], st["qrope"], st["pool"], st["tables"], None, st["rows"], st["n_rows"], b,
                                st["h"], k, st["blocks"], KVL, ROPE, PT, n_pages, W ** -0.5, st["precise"], st["clat"],
                                st["partial"], None, s)
    return st["scores"], st["rows"], st["clat"]


# ---- attention -----------------------------------------------------------------------------

def _prepare_attend(case, mk):
    lens = _lens(case)
    b, h = case["batch"], case["heads"]
    blocks, top = -(-case["ctx"] // PT), int(lens.max())
    tables = mk.tables(b, blocks)
    pool, _ = _filled_pool(mk, tables, lens)
    return dict(b=b, h=h, top=top, blocks=blocks, tables=tables, pool=pool, n_pages=b * blocks,
                precise=case["precise"], lens=torch.from_numpy(lens).cuda(), slots=_next_slots(tables, lens),
                new=mk.normal(b, W).bfloat16(), qabs=mk.normal(b, h, KVL), qrope=mk.normal(b, h, ROPE),
                clat=_empty(b, h, KVL), partial=_empty(max(hip.mla_attend_paged_scratch_floats(b, h, top), 4)))


def _run_attend(st, s):
    hip.launch_kv_append_paged(st["new"], st["slots"], st["pool"], st["b"], W, PT, st["n_pages"], None, s)
    hip.launch_mla_attend_paged(st["qabs"], st["qrope"], st["pool"], st["tables"], st["lens"], None, None, st["b"],
                                st["h"], st["top"], st["blocks"], KVL, ROPE, PT, st["n_pages"], W ** -0.5,
                                st["precise"], st["clat"], st["partial"], None, s)
    return st["clat"]


# ---- the single-sequence engine over linear slabs ------------------------------------------

def _prepare_engine(case, mk):
    nt, h, nb = case["nt"], case["heads"], KVL // 128
    k = min(case["k"], nt)
    lc8, lscale = _zeros(nt, KVL, dtype=torch.uint8), _zeros(nt, nb)
    rc, kcache = _zeros(nt, ROPE, dtype=torch.bfloat16), mk.normal(nt, INDEX_DIM).bfloat16()
    hip.launch_append_kv_rows(mk.normal(nt, KVL), mk.normal(nt, ROPE), lc8, lscale, rc, 0, nt, KVL, ROPE, nb)
    return dict(nt=nt, k=k, h=h, nb=nb, lc8=lc8, lscale=lscale, rc=rc, kcache=kcache, latent=mk.normal(KVL),
                rope=mk.normal(ROPE), key=mk.normal(INDEX_DIM), iq=mk.normal(INDEX_HEADS, INDEX_DIM),
                iw=mk.uniform(INDEX_HEADS), scores=_zeros(nt), rows=_zeros(k, dtype=torch.int32),
                qabs=mk.normal(h, KVL), qrope=mk.normal(h, ROPE), clat=_empty(h, KVL),
                partial=_empty(hip.attend_scratch_floats(h, KVL)))


def _run_engine(st, s):
    nt, k, h, nb = st["nt"], st["k"], st["h"], st["nb"]
    hip.launch_append_kv(st["latent"], st["rope"], st["lc8"], st["lscale"], st["rc"], nt - 1, KVL, ROPE, nb)
    hip.launch_index_append(st["key"], st["kcache"], nt - 1, INDEX_DIM)
    hip.launch_index_score(st["iq"], st["iw"], st["kcache"], None, nt, INDEX_HEADS, INDEX_HEADS, INDEX_DIM,
                           INDEX_DIM ** -0.5, 1.0, st["scores"])
    hip.launch_index_topk(st["scores"], nt, k, st["rows"])
    hip.launch_attend(st["qabs"], st["qrope"], st["lc8"], st["lscale"], st["rc"], st["rows"], h, k, KVL, ROPE, nb,
                      W ** -0.5, st["clat"], st["partial"])
    return st["scores"], st["rows"], st["clat"]


# ---- the second cache format ---------------------------------------------------------------

def _rotation(n, rd):
    """(cos, sin) pairs of the compressed rotation table for n positions."""
    inv = 160000.0 ** (-torch.arange(rd // 2, device="cuda", dtype=torch.float64) * 2.0 / rd)
    ang = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * inv[None, :]
    return torch.stack([torch.cos(ang), torch.sin(ang)], dim=-1).reshape(n, rd).float().contiguous()


class _Compressor:
    """A compressor's weights and its window state, holding the tokens before the next one."""

    def __init__(self, mk, ratio, d, rd, positions):
        self.geom = hip.CompGeom.build(ratio, d, rd, V4_EPS)
        self.ape, self.norm = mk.normal(ratio, self.geom.cd), 1.0 + 0.1 * mk.normal(d)
        self.freqs = _rotation(positions, rd)
        n = self.geom.coff * ratio
        self.kv_state, self.score_state = mk.normal(n, self.geom.cd), 2.0 * mk.normal(n, self.geom.cd)


def _prepare_v4_cache(case, mk):
    n, ratio = case["tokens"], case["ratio"]
    comp, n_comp = _Compressor(mk, ratio, V4_DIM, V4_DIM - V4_QUANT, n), n // ratio
    # the prompt's rows, then the pooled rows: what the prompt's attention indexes
    src, kv = mk.rows(n, V4_DIM, 0.01, 200.0).bfloat16().float(), _zeros(n + n_comp, V4_DIM)
    kv[:n] = src
    st = dict(n=n, n_comp=n_comp, ratio=ratio, comp=comp, kv=kv, ring=_zeros(V4_WINDOW, V4_DIM),
              ckv=mk.normal(n, comp.geom.cd), cscore=2.0 * mk.normal(n, comp.geom.cd))
    if n_comp:
        st["fin"] = hip.CompFinish.of(comp.norm, comp.freqs, kv[n:])
    return st


def _run_v4_cache(st, s):
    n, n_comp, comp, kv = st["n"], st["n_comp"], st["comp"], st["kv"]
    hip.launch_act_quant_f8_prefix(kv, kv, n, V4_DIM, V4_QUANT, V4_BLOCK, s)
    hip.launch_kv_ring_write(kv, st["ring"], V4_WINDOW, V4_DIM, n, 0, s)
    hip.launch_kv_compress_deposit(st["ckv"], st["cscore"], comp.ape, comp.kv_state, comp.score_state, comp.geom, n, 0, s)
    if n_comp:
        hip.launch_kv_compress_prefill(st["ckv"], st["cscore"], comp.ape, st["fin"], comp.geom, n_comp, s)
        pooled = kv.data_ptr() + n * V4_DIM * 4
        hip.launch_act_quant_f8_prefix(pooled, pooled, n_comp, V4_DIM, V4_QUANT, V4_BLOCK, s)
    return kv, st["ring"], comp.kv_state, comp.score_state


def _index_inputs(mk, n, n_comp):
    """The indexer's queries before their spread, its compressor's finished rows, the head weights."""
    kv = mk.normal(n_comp, INDEX_DIM).bfloat16().float()
    hip.launch_act_quant_f4_rotated(kv, n_comp, INDEX_DIM)
    return dict(iq=mk.normal(n * INDEX_HEADS, INDEX_DIM).bfloat16().float(), ikv=kv,
                iw=(mk.normal(n, INDEX_HEADS) * INDEX_DIM ** -0.5).bfloat16().float())


def _prepare_v4_index(case, mk):
    n = case["tokens"]
    n_comp = n // V4_RATIO
    cols = min(n, V4_WINDOW) + min(V4_CAP, n_comp)
    return dict(_index_inputs(mk, n, n_comp), n=n, n_comp=n_comp, scores=_zeros(n, n_comp),
                sel=_zeros(n, cols, dtype=torch.int32))


def _run_v4_index(st, s):
    n, n_comp = st["n"], st["n_comp"]
    hip.launch_act_quant_f4_rotated(st["iq"], n * INDEX_HEADS, INDEX_DIM, s)
    hip.launch_index_score_blocks_prefill(st["iq"], st["ikv"], st["iw"], st["scores"], n, n_comp, INDEX_HEADS,
                                          INDEX_DIM, V4_RATIO, s)
    hip.launch_sel_gather_scored(st["scores"], n_comp, V4_WINDOW, V4_RATIO, V4_CAP, n, 0, st["sel"], s)
    return st["iq"], st["scores"], st["sel"]


def _cache_rows(mk, n):
    """Rows as the cache holds them: simulated fp8 in the first 448 dims, bf16 after."""
    kv = mk.rows(n, V4_DIM, 0.01, 20.0).bfloat16().float()
    hip.launch_act_quant_f8_prefix(kv, kv, n, V4_DIM, V4_QUANT, V4_BLOCK)
    return kv


def _prepare_v4_attend(case, mk):
    n = case["tokens"]
    n_comp = n // V4_RATIO
    cols = min(n, V4_WINDOW) + min(V4_CAP, n_comp)
    idx = _zeros(n, cols, dtype=torch.int32)
    hip.launch_sel_gather_scored(mk.normal(n, n_comp), n_comp, V4_WINDOW, V4_RATIO, V4_CAP, n, 0, idx)
    return dict(n=n, cols=cols, idx=idx, kv=_cache_rows(mk, n + n_comp), sink=mk.normal(V4_HEADS),
                q=mk.normal(n, V4_HEADS, V4_DIM).bfloat16().float(), o=_empty(n, V4_HEADS, V4_DIM))


def _run_v4_attend(st, s):
    hip.launch_gather_attn_shared_kv(st["q"], st["kv"], st["sink"], st["idx"], st["n"], V4_HEADS, V4_DIM, st["cols"],
                                     V4_DIM ** -0.5, st["o"], s)
    return st["o"]


def _prepare_v4_decode(case, mk):
    pos = case["pos"]
    n_comp = (pos + 1) // V4_RATIO
    cols = V4_WINDOW + min(V4_CAP, n_comp)
    attn = _Compressor(mk, V4_RATIO, V4_DIM, V4_DIM - V4_QUANT, pos + 1)
    indexer = _Compressor(mk, V4_RATIO, INDEX_DIM, 64, pos + 1)
    cache = _cache_rows(mk, V4_WINDOW + n_comp)
    st = dict(_index_inputs(mk, 1, n_comp), pos=pos, n_comp=n_comp, cols=cols, attn=attn, indexer=indexer, cache=cache,
              entry=mk.normal(1, V4_DIM).bfloat16().float(), ckv=mk.normal(1, attn.geom.cd),
              cscore=2.0 * mk.normal(1, attn.geom.cd), xkv=mk.normal(1, indexer.geom.cd),
              xscore=2.0 * mk.normal(1, indexer.geom.cd), scores=_zeros(n_comp), idx=_zeros(cols, dtype=torch.int32),
              sink=mk.normal(V4_HEADS), q=mk.normal(V4_HEADS, V4_DIM).bfloat16().float(), o=_empty(V4_HEADS, V4_DIM),
              partial=_empty(max(hip.gather_attn_scratch_floats(1, V4_HEADS, V4_DIM, cols), 4)))
    dst = hip.compress_dst(V4_RATIO, V4_WINDOW, 1, pos)
    if dst is not None:                      # this position closes a block: its rows' homes
        st["row"], st["xrow"] = cache[dst[0]:], st["ikv"][pos // V4_RATIO:]
        st["fin"] = hip.CompFinish.of(attn.norm, attn.freqs, st["row"])
        st["xfin"] = hip.CompFinish.of(indexer.norm, indexer.freqs, st["xrow"])
    return st


def _run_v4_decode(st, s):
    pos, n_comp, attn, indexer, cache = st["pos"], st["n_comp"], st["attn"], st["indexer"], st["cache"]
    hip.launch_act_quant_f8_prefix(st["entry"], st["entry"], 1, V4_DIM, V4_QUANT, V4_BLOCK, s)
    hip.launch_kv_ring_write(st["entry"], cache, V4_WINDOW, V4_DIM, 1, pos, s)
    slot = pos % V4_RATIO
    hip.launch_kv_compress_deposit(st["ckv"], st["cscore"], attn.ape, attn.kv_state, attn.score_state, attn.geom, 1, slot, s)
    hip.launch_kv_compress_deposit(st["xkv"], st["xscore"], indexer.ape, indexer.kv_state, indexer.score_state,
                                   indexer.geom, 1, slot, s)
    if "fin" in st:
        hip.launch_kv_compress_decode(attn.kv_state, attn.score_state, st["fin"], attn.geom, pos, s)
        hip.launch_act_quant_f8_prefix(st["row"], st["row"], 1, V4_DIM, V4_QUANT, V4_BLOCK, s)
        hip.launch_kv_compress_decode(indexer.kv_state, indexer.score_state, st["xfin"], indexer.geom, pos, s)
        hip.launch_act_quant_f4_rotated(st["xrow"], 1, INDEX_DIM, s)
    hip.launch_act_quant_f4_rotated(st["iq"], INDEX_HEADS, INDEX_DIM, s)
    hip.launch_index_score_blocks(st["iq"], st["ikv"], st["iw"], st["scores"], 1, n_comp, INDEX_HEADS, INDEX_DIM, s)
    hip.launch_sel_gather_scored(st["scores"], n_comp, V4_WINDOW, V4_RATIO, V4_CAP, 1, pos, st["idx"], s)
    hip.launch_gather_attn_shared_kv(st["q"], cache, st["sink"], st["idx"], 1, V4_HEADS, V4_DIM, st["cols"],
                                     V4_DIM ** -0.5, st["o"], s, n_kv=V4_WINDOW + n_comp, partial=st["partial"])
    return st["o"], st["idx"], st["scores"], cache, st["ikv"], attn.kv_state, attn.score_state
