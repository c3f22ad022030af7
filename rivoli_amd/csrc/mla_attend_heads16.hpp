// MLA decode attention for calls that the 64-head workgroups of mla_attend.hip leave most of the
// chip idle on, or keep for a few tiles only: the same arithmetic (bf16 matrix instructions, q
// and the weights as bf16 hi + lo in the parity mode), dealt the other way. Included by
// mla_attend.hip. Long work items of few heads take it (heads16_few); the others, and the linear slabs, take
// mla_attend_few.hpp, which came later: figures of other calls here are from before that.
//
// There a workgroup's eight waves share one tile: two of them meet in LDS over every score, and
// a barrier ends every tile. A short call is then a chain — list entry, table, rows, staging,
// exchange, barrier, softmax — walked a few times by a few workgroups. Here a workgroup owns 16
// heads, and each of its four waves (one per SIMD, each with the whole register file) walks
// 32-token tiles of its own from memory to accumulators without meeting another wave: 128 tokens
// are in work at a time, four times as many workgroups share a call's tokens for the same
// partial records, and the only barriers are around the query and the merge of the four waves'
// results at the end.
//
// A wave's rows go from memory straight into LDS as they are (global_load_lds, two buffers) and
// become bf16 when an operand is read: four conversions per eight values on either side, but a
// quarter of the LDS traffic of a tile staged as bf16, which is what a first form of this kernel
// was bound by (16 heads use a tile a quarter as often as 64 do).
// Measured, parity mode, 64 heads, with the merge of the records: one sequence of 4 096 tokens
// 34.5 -> 21 us, 8 x 2 048 listed rows 38 -> 24 us. A wave of two listed tiles lives 39 500 cycles, by counter: matrix instructions (272)
// 4 350, vector instructions 11 700, waits 17 100 (the first rows, the merge), the rest transfers, LDS and
// scalar instructions.
#pragma once

namespace rk {

constexpr int kH16Threads = kH16Waves * kWave;
constexpr int kH16ColTiles = kKvl / 16;
constexpr int kH16Chunks = kKSteps / 2;  // 16-byte pieces of a row per lane group: two K-steps each

// A wave's tile in LDS: rows of codes with one 16-byte granule of padding, so that sixteen rows'
// 16-byte reads meet in no bank, and the second sixteen rows 128 bytes further on, so that the
// transposing reads, which take rows r and r + 16 together, do not either.
struct H16Tile {
    static constexpr int kGranules = kRowW / 16 + 1;  // of a row
    static constexpr int kRow = kGranules * 16;
    static constexpr int kGap = 8;                    // granules between the halves
    static constexpr int kAll = kTile * kGranules + kGap;
    static constexpr int kBytes = kAll * 16;
    static constexpr int kRequests = (kAll + kWave - 1) / kWave;
    static constexpr int kWaveBytes = 2 * kBytes;
    static __device__ __forceinline__ int at(int row) { return row * kRow + (row >> 4) * (kGap * 16); }
};
static_assert(kH16ColTiles * kWave * 16 <= 2 * H16Tile::kBytes, "a wave's accumulators pass through its tiles' room");
static_assert(5 * 2048 <= H16Tile::kBytes, "five K-steps of the query's operands fit a second buffer");

// One part of a workgroup's work, as attend_part: rows [r_begin, r_end) of sequence `seq`, heads
// 16 * hg .. +15.
template <int QSPLIT, int PSPLIT, int MODE>
__device__ __forceinline__ void attend_part_heads16(const AttendArgs& a, int seq, int hg, int r_begin, int r_end,
                                                    bool whole, float* pa, float* pml) {
    static_assert(MODE == kDense || MODE == kSparse, "paged rows, looked up one by one");
    using T = H16Tile;
    __shared__ __attribute__((aligned(16))) uint8_t smem[kH16Waves * T::kWaveBytes];
    __shared__ __attribute__((aligned(16))) float token_scale[kH16Waves][kTile];
    __shared__ float wave_ml[kH16Waves][kH16Heads][2];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, n16 = lane & 15;
    const int n_tiles = (r_end - r_begin + kTile - 1) / kTile;
    const lds_ptr<uint8_t> room = (lds_ptr<uint8_t>)smem;
    const lds_ptr<uint8_t> own = room + wave * T::kWaveBytes;
    const lds_ptr<float> scl_lds = (lds_ptr<float>)token_scale[wave];

    // ---- where a tile's rows are: lane r < 32 resolves row r ----------------------------------
    constexpr unsigned long long kNone = ~0ull;
    const unsigned int* const rows_g = MODE == kSparse ? a.rows + (size_t)seq * a.k : nullptr;
    const int* const table_g = a.block_table + (size_t)seq * a.max_blocks;
    // the list entry (or position) of the lane's row; the read is unconditional and clamped
    auto token_of = [&](int tile) -> unsigned int {
        // (unsigned: three rounds of tiles past the end of 2^31 - 32 rows is past what an int holds)
        const unsigned int pos = min((unsigned)r_begin + (unsigned)tile * kTile + (lane & 31), (unsigned)r_end - 1u);
        return rows_g ? rows_g[pos] : pos;
    };
    // the row's page, likewise (-1: the block table has no entry for it)
    auto page_of = [&](unsigned int tok) -> int {
        const unsigned int blk = a.page_shift >= 0 ? tok >> a.page_shift : tok / (unsigned)a.page_tokens;
        const int page = table_g[min(blk, (unsigned)a.max_blocks - 1)];
        return blk < (unsigned)a.max_blocks ? page : -1;
    };
    struct Where {
        unsigned long long code, scale;
    };
    auto resolve = [&](int tile, unsigned int tok, int page) -> Where {
        Where w = {kNone, 0};
        if (lane >= kTile || tile >= n_tiles || r_begin + tile * kTile + lane >= r_end) return w;
        // a list entry of all ones is nobody's token, and only the 8-bit modes count it (as attend_part)
        if (MODE != kDense && tok == 0xffffffffu && !a.count_ones) return w;
        if ((unsigned)page < (unsigned)a.n_pages) {
            const unsigned int off =
                a.page_shift >= 0 ? tok & (unsigned)(a.page_tokens - 1) : tok % (unsigned)a.page_tokens;
            const unsigned long long base = (unsigned long long)page * a.page_bytes;
            w.code = base + (unsigned long long)off * kRowW;
            w.scale = base + (unsigned long long)a.page_tokens * kRowW + (unsigned long long)off * 4;
        } else if (a.bad_rows && hg == 0) {
            atomicAdd(a.bad_rows, 1u);
        }
        return w;
    };

    // ---- a tile on its way into LDS -------------------------------------------------------------
    // Request i fills granules 64 i .. +63 of the tile; `from` packs, per request, the row a lane's
    // granule belongs to and its place in the row (the padding and the gap repeat a neighbour).
    uint32_t from[T::kRequests];
#pragma unroll
    for (int i = 0; i < T::kRequests; ++i) {
        int gi = kWave * i + lane;
        gi = gi < 16 * T::kGranules ? gi : max(gi - T::kGap, 16 * T::kGranules - 1);
        const int row = min(gi / T::kGranules, kTile - 1), c = min(gi - row * T::kGranules, T::kGranules - 2);
        from[i] = (uint32_t)row | (uint32_t)(16 * c) << 8;
    }
    unsigned int there_next = 0;      // bit r: row r of the requested tile exists
    float scale_next = 0.0f;          // lanes 0..31: its scale
    auto request = [&](const Where& w, int buf) {
        there_next = (unsigned int)__builtin_amdgcn_ballot_w64(w.code != kNone);
        const unsigned long long at = w.code != kNone ? w.code : 0;  // a row that is not there reads the first one
        const uint32_t lo = (uint32_t)at, hi = (uint32_t)(at >> 32);
        // (scalar by construction: the transfer takes its LDS base from a scalar register)
        const lds_ptr<uint8_t> to = (lds_ptr<uint8_t>)(uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane(
            (int)(uint32_t)(uintptr_t)(own + buf * T::kBytes));
#pragma unroll
        for (int i = 0; i < T::kRequests; ++i) {
            const int row = (int)(from[i] & 0xffu);
            const unsigned long long b = ((unsigned long long)(uint32_t)__shfl((int)hi, row, kWave) << 32) | (uint32_t)__shfl((int)lo, row, kWave);
            if (kWave * (i + 1) <= T::kAll || lane < T::kAll - kWave * i)
                dma16(a.pool + b + (from[i] >> 8), to + 1024 * i);
        }
        scale_next = *reinterpret_cast<const float*>(a.pool + w.scale);
    };

    // ---- prologue -------------------------------------------------------------------------------
    // The wave's first tile is looked up and requested, then the query: each wave turns every
    // fourth K-step of the 16 heads into operands, all waves read all of them from LDS.
    unsigned int tok0 = token_of(wave), tok1 = token_of(wave + kH16Waves), tok2 = token_of(wave + 2 * kH16Waves);
    const int head = hg * kH16Heads + n16;
    // dims of K-step j, lane group g: eight from dim_of(j). A lane's two K-steps 2c, 2c + 1 are one
    // 16-byte piece of a row. The pieces of lane groups 0, 1 (and 2, 3), read together, lie
    // 256 bytes apart, in the same banks of different rows.
    auto dim_of = [&](int j) -> int {
        const int c = j >> 1, s = j & 1;
        if (c == 8) return kKvl + 16 * g + 8 * s;
        return 256 * (g & 1) + 128 * (g >> 1) + 16 * c + 8 * s;
    };
    constexpr int kMine = (kKSteps + kH16Waves - 1) / kH16Waves;
    float4 qv[kMine][2];
    {
        const size_t qrow = (size_t)seq * a.H + (head < a.H ? head : 0);
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            const int d = dim_of(min(wave + m * kH16Waves, kKSteps - 1));
            const float* src = d < kKvl ? a.qabs + qrow * kKvl + d : a.qrope + qrow * kRopeW + (d - kKvl);
            qv[m][0] = reinterpret_cast<const float4*>(src)[0], qv[m][1] = reinterpret_cast<const float4*>(src)[1];
        }
    }
    int page1 = page_of(tok1);
    request(resolve(wave, tok0, page_of(tok0)), 0);
    // the operands pass through the waves' second buffers, five K-steps each
    auto q_room = [&](int j) -> lds_ptr<uint8_t> {
        return room + (j / 5) * T::kWaveBytes + T::kBytes + (j % 5) * 2048 + 16 * lane;
    };
    {
        const float keep = head < a.H ? a.qscale : 0.0f;
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            const int j = wave + m * kH16Waves;
            if (j >= kKSteps) break;  // wave-uniform
            const float v[8] = {qv[m][0].x, qv[m][0].y, qv[m][0].z, qv[m][0].w, qv[m][1].x, qv[m][1].y, qv[m][1].z, qv[m][1].w};
            bf16x8 hi, lo;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float x = v[i] * keep;
                hi[i] = (__bf16)x;
                lo[i] = (__bf16)(x - (float)hi[i]);
            }
            *(lds_ptr<bf16x8>)q_room(j) = hi;
            if (QSPLIT == 2) *(lds_ptr<bf16x8>)(q_room(j) + 1024) = lo;
        }
    }
    __syncthreads();
    bf16x8 qh[kKSteps], ql[QSPLIT == 2 ? kKSteps : 1];
#pragma unroll
    for (int j = 0; j < kKSteps; ++j) {
        qh[j] = *(lds_ptr<bf16x8>)q_room(j);
        if (QSPLIT == 2) ql[j] = *(lds_ptr<bf16x8>)(q_room(j) + 1024);
    }
    __syncthreads();  // the second buffers are the tiles' from here on

    f32x4 o[kH16ColTiles];
#pragma unroll
    for (int nt = 0; nt < kH16ColTiles; ++nt) o[nt] = f32x4{0, 0, 0, 0};
    float m_ref = -INFINITY, l_sum = 0.0f;

    int buf = 0;
    for (int tile = wave; tile < n_tiles; tile += kH16Waves, buf ^= 1) {
        // Everything asked for has landed: this tile (asked for a whole tile's work ago) and the
        // lookups for the next two. The values the compiler tracks are used here, where nothing is
        // in flight, so that it has nothing to wait for later: its waits would cover the transfers.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("" : "+v"(tok1), "+v"(tok2), "+v"(page1), "+v"(scale_next));
        const lds_ptr<uint8_t> codes = own + buf * T::kBytes;
        const unsigned int here = there_next;
        if (lane < kTile) {
            // a scale that is not a positive number cannot come from the append: such a token is
            // left out like one that is not there
            scl_lds[lane] = ((here >> lane) & 1u) && scale_next > 0.0f ? scale_next : 0.0f;
        }
        // rows that are not there: their codes must be finite, they meet a zero weight
        for (unsigned int gone = ~here; gone; gone &= gone - 1)
            if (lane < T::kGranules) *(lds_ptr<u32x4>)(codes + T::at(__builtin_ctz(gone)) + 16 * lane) = u32x4{0, 0, 0, 0};
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // LDS serves a wave in order: for the compiler
        if (tile + kH16Waves < n_tiles) request(resolve(tile + kH16Waves, tok1, page1), buf ^ 1);
        tok1 = tok2;
        page1 = page_of(tok1);
        tok2 = token_of(tile + 3 * kH16Waves);

        // ---- scores: S^T[token][head], two 16-token halves ------------------------------------
        f32x4 s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
        // the lane's tokens' scales: 4g + i, 16 + 4g + i
        const f32x4 sa = *(lds_ptr<f32x4>)(scl_lds + 4 * g), sb = *(lds_ptr<f32x4>)(scl_lds + 16 + 4 * g);
        const lds_ptr<uint8_t> a0p = codes + T::at(n16), a1p = codes + T::at(16 + n16);
        auto as_bf16 = [](uint32_t x, uint32_t y) -> bf16x8 {
            u32x4 d;
            uint32_t d0, d1, d2, d3;
            e4m3x4_to_bf16(x, d0, d1);
            e4m3x4_to_bf16(y, d2, d3);
            d = u32x4{d0, d1, d2, d3};
            return __builtin_bit_cast(bf16x8, d);
        };
        auto step = [&](int j, bf16x8 f0, bf16x8 f1) {
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f0, qh[j], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f1, qh[j], s1, 0, 0, 0);
            if (QSPLIT == 2) {
                s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f0, ql[j], s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f1, ql[j], s1, 0, 0, 0);
            }
        };
        u32x4 c0[2], c1[2];
        c0[0] = *(lds_ptr<u32x4>)(a0p + dim_of(0)), c1[0] = *(lds_ptr<u32x4>)(a1p + dim_of(0));
#pragma unroll
        for (int c = 0; c < kH16Chunks; ++c) {
            if (c + 1 < kH16Chunks) {
                c0[(c + 1) & 1] = *(lds_ptr<u32x4>)(a0p + dim_of(2 * c + 2));
                c1[(c + 1) & 1] = *(lds_ptr<u32x4>)(a1p + dim_of(2 * c + 2));
            }
            __builtin_amdgcn_sched_barrier(0);
            const u32x4 x = c0[c & 1], y = c1[c & 1];
            step(2 * c, as_bf16(x.x, x.y), as_bf16(y.x, y.y));
            step(2 * c + 1, as_bf16(x.z, x.w), as_bf16(y.z, y.w));
            __builtin_amdgcn_sched_barrier(0);
        }

        // The first value-side operands come out of LDS under the softmax. Operand of column tile
        // nt: the transposing load hands a lane the codes of column 16 nt + n16 for its eight
        // tokens, 4g + e and 16 + 4g + e; source lane pair e addresses token e's row.
        const int e8 = n16 >> 1;
        const lds_ptr<uint8_t> vrow = codes + T::at(16 * (e8 >> 2) + 4 * g + (e8 & 3)) + 8 * (n16 & 1);
        constexpr int kValueAhead = 4;
        i32x2 fb[2][kValueAhead];
#pragma unroll
        for (int i = 0; i < kValueAhead; ++i) fb[0][i] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr<i32x2>)(vrow + 16 * i));
        __builtin_amdgcn_sched_barrier(0);

        // ---- online softmax over the lane's 8 tokens of head n16 (attend_part's) ------------------
        float v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = sa[i] > 0.0f ? s0[i] * sa[i] : -INFINITY;
            v[4 + i] = sb[i] > 0.0f ? s1[i] * sb[i] : -INFINITY;
        }
        float tmax = fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmaxf(fmaxf(v[4], v[5]), fmaxf(v[6], v[7])));
        tmax = rows_max(tmax);
        const bool grow = tmax > m_ref + kLazyRescale;  // false while nothing is there
        const float corr = grow ? __builtin_amdgcn_exp2f(m_ref - tmax) : 1.0f;  // 2^-inf = 0 at first
        // (accumulators that are still zero need no rescaling: the first tile's, always)
        if (__builtin_amdgcn_ballot_w64(grow && m_ref != -INFINITY) != 0) {
            float c[4];  // the lane's accumulators are heads 4g+i; corr lives in lanes n16 == head
#pragma unroll
            for (int i = 0; i < 4; ++i) c[i] = __shfl(corr, 4 * g + i, kWave);
#pragma unroll
            for (int nt = 0; nt < kH16ColTiles; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[nt][i] *= c[i];
        }
        if (grow) m_ref = tmax;
        l_sum *= corr;
        const float mu = m_ref == -INFINITY ? 0.0f : m_ref;
        // the weights under their tokens' scales
        bf16x8 p, p_lo;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float e = __builtin_amdgcn_exp2f(v[i] - mu);  // not there -> 0
            const float scl = i < 4 ? sa[i & 3] : sb[i & 3];
            const float x = e * scl;
            const __bf16 w = (__bf16)x;
            p[i] = w;
            if (PSPLIT == 2) {
                p_lo[i] = (__bf16)(x - (float)w);
                l_sum += e;
            } else {
                l_sum += (float)w * (scl > 0.0f ? __builtin_amdgcn_rcpf(scl) : 0.0f);
            }
        }

        // ---- values: O[head][col] += P . V ----------------------------------------------------
#pragma unroll
        for (int n0 = 0; n0 < kH16ColTiles; n0 += kValueAhead) {
            const int cur = (n0 / kValueAhead) & 1;
            if (n0 + kValueAhead < kH16ColTiles) {
#pragma unroll
                for (int i = 0; i < kValueAhead; ++i)
                    fb[cur ^ 1][i] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr<i32x2>)(vrow + 16 * (n0 + kValueAhead + i)));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kValueAhead; ++i) {
                const bf16x8 f = as_bf16((uint32_t)fb[cur][i][0], (uint32_t)fb[cur][i][1]);
                o[n0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p, f, o[n0 + i], 0, 0, 0);
                if (PSPLIT == 2) o[n0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p_lo, f, o[n0 + i], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // a wave without a tile has a request of its own in flight

    // ---- the four waves' results become one: accumulators under the common maximum, summed in
    // wave order, each wave a quarter of the columns ------------------------------------------------
    l_sum = rows_sum(l_sum);
    if (g == 0) wave_ml[wave][n16][0] = m_ref, wave_ml[wave][n16][1] = l_sum;
    __syncthreads();
    float m_all = -INFINITY, l_all = 0.0f;
#pragma unroll
    for (int w = 0; w < kH16Waves; ++w) m_all = fmaxf(m_all, wave_ml[w][n16][0]);
#pragma unroll
    for (int w = 0; w < kH16Waves; ++w) {
        const float m_w = wave_ml[w][n16][0];
        if (m_w != -INFINITY) l_all += wave_ml[w][n16][1] * __builtin_amdgcn_exp2f(m_w - m_all);
    }
    const float mine = m_ref == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_ref - m_all);
    float c[4], l_h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = __shfl(mine, 4 * g + i, kWave), l_h[i] = __shfl(l_all, 4 * g + i, kWave);
#pragma unroll
    for (int nt = 0; nt < kH16ColTiles; ++nt)
        *(lds_ptr<f32x4>)(own + (nt * kWave + lane) * 16) =
            f32x4{o[nt][0] * c[0], o[nt][1] * c[1], o[nt][2] * c[2], o[nt][3] * c[3]};
    __syncthreads();
    constexpr int kShare = kH16ColTiles / kH16Waves;
    const int h0 = hg * kH16Heads + 4 * g;
    float* const dst = (whole ? a.clat + (size_t)seq * a.H * kKvl : pa) + (size_t)h0 * kKvl + 16 * kShare * wave + n16;
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = !whole ? 1.0f : l_h[i] > 0.0f ? 1.0f / l_h[i] : 0.0f;
#pragma unroll
    for (int u = 0; u < kShare; ++u) {
        const lds_ptr<uint8_t> at = room + ((wave * kShare + u) * kWave + lane) * 16;
        f32x4 sum = *(lds_ptr<f32x4>)at;
#pragma unroll
        for (int w = 1; w < kH16Waves; ++w) sum += *(lds_ptr<f32x4>)(at + w * T::kWaveBytes);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (h0 + i < a.H) dst[i * kKvl + 16 * u] = sum[i] * c[i];
    }
    if (!whole && wave == 0 && g == 0 && head < a.H) {
        pml[head * 2] = m_all;
        pml[head * 2 + 1] = l_all;
    }
}

}  // namespace rk
