// MLA decode attention by workgroups of 32 heads, eight waves on one 64-token tile: mla_attend_few.hpp's
// pipeline (its transfers, two barriers a tile, records) over twice the heads, for calls whose work items are long enough
// to be worth half as many head groups (heads32_pays). Included by mla_attend.hip.
//
// A tile there is bound by its chain and by what does not depend on the heads: 68 conversions of codes a wave, its
// lookups and transfers, two barriers. Here all of that serves 32 heads. Matrix tiles are 32 x 32: a wave has 32
// tokens' scores over a quarter of the dims (so that its query operands still are 72 registers), four heads' softmax (four tokens
// a lane) and 64 columns of the values. Four partial scores meet in LDS, 34 KB of it: with three tiles of codes the whole 160 KB, so
// a tile's roped keys share their 128-byte groups between two waves' rows, and the calls are those that SeqDeal cuts, which
// needs no table of the sequences.
#pragma once

namespace rk {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWideWaves = 8;
constexpr int kWideThreads = kWideWaves * kWave;
constexpr int kWideTokens = 64;                            // of a tile
constexpr int kWideSteps = 9;                              // a wave's K-steps of 16 dims: eight of its 128 latent dims, one roped
constexpr int kWideBuffers = 3;
// A tile in LDS: 4 KB of each wave, its eight rows' codes in four groups of 128 bytes, a group's rows next to each other; then 1 KB of roped
// codes for each two waves. A row's eight 16-byte pieces of a group change places by the row's number, (row >> 1) & 7, so that reads of one
// piece of sixteen rows meet in no bank; the rows of the even wave of two have their four roped pieces in the lower 64 bytes then, those
// of the odd one in the upper.
constexpr int kWideRopeAt = kWideWaves * 4096;
constexpr int kWideTileBytes = kWideRopeAt + kWideWaves / 2 * 1024;
constexpr int kWideScoreStride = kWideTokens + 4;
constexpr int kWideInFlight = 6;                           // a tile's transfers by a wave, after its lookups
static_assert(kRowW == 576 && kKvl == 512, "four quarters of 128 latent and 16 roped dims");

template <int QSPLIT, int PSPLIT, int MODE>
__device__ __forceinline__ void attend_part_wide(const AttendArgs& a, int seq, int hg, int r_begin, int r_end,
                                                 bool whole, float* pa, float* pml) {
    static_assert(MODE == kDense || MODE == kSparse, "paged rows, looked up one by one");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[kWideBuffers * kWideTileBytes];
    __shared__ __attribute__((aligned(16))) float score_smem[4 * kWideHeads * kWideScoreStride];
    __shared__ __attribute__((aligned(16))) uint8_t weight_smem[PSPLIT * kWideHeads * kWideTokens * 2];
    __shared__ __attribute__((aligned(16))) float scale_smem[2][kWideTokens];  // by the tile's parity
    __shared__ __attribute__((aligned(16))) float scale_raw[kWideBuffers][kWideWaves][kWave];
    // a tile's list entries and pages, 8 a wave, by the tile's number
    __shared__ __attribute__((aligned(16))) unsigned int token_smem[4][kWideWaves][8];
    __shared__ __attribute__((aligned(16))) int page_smem[4][kWideWaves][8];
    __shared__ float corr_smem[kWideHeads], ml_smem[kWideHeads][2];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5, n32 = lane & 31;
    const int n_tiles = (r_end - r_begin + kWideTokens - 1) / kWideTokens;
    const lds_ptr<uint8_t> rows = (lds_ptr<uint8_t>)smem;
    const lds_ptr<float> scores = (lds_ptr<float>)score_smem;
    const lds_ptr<uint8_t> weights = (lds_ptr<uint8_t>)weight_smem;

    // ---- where a tile's rows are: eight lanes ask for row 8 wave + (lane >> 3) (as attend_part_few) ------------
    const int my_row = 8 * wave + (lane >> 3), l8 = lane & 7;
    const unsigned int* const rows_g = MODE == kSparse ? a.rows + (size_t)seq * a.k : nullptr;
    const int* const table_g = a.block_table + (size_t)seq * a.max_blocks;
    auto at_of = [&](int tile, int row) -> unsigned int {  // clamped: lookups run past the end
        return min((unsigned)r_begin + (unsigned)tile * kWideTokens + (unsigned)row, (unsigned)r_end - 1u);
    };
    auto token_of = [&](int tile, int row) -> unsigned int {
        const unsigned int at = at_of(tile, row);
        return rows_g ? rows_g[at] : at;
    };
    auto block_of = [&](unsigned int tok) -> unsigned int {
        return a.page_shift >= 0 ? tok >> a.page_shift : tok / (unsigned)a.page_tokens;
    };
    auto entry_of = [&](unsigned int tok) -> const int* { return table_g + min(block_of(tok), (unsigned)a.max_blocks - 1); };

    // ---- a tile on its way into LDS ----------------------------------------------------------------------------
    auto scalar = [](lds_ptr<uint8_t> p) -> lds_ptr<uint8_t> {  // the transfers take their LDS base from a scalar register
        return (lds_ptr<uint8_t>)(uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)p);
    };
    const int swap = (4 * (wave & 1) + (lane >> 4)) & 7;  // (my_row >> 1) & 7
    const unsigned long long roped = __builtin_amdgcn_ballot_w64(16 * (l8 ^ swap) < kRopeW);  // lanes with a piece of the roped codes
    auto request = [&](int tile, int buf, unsigned int tok, int page) -> bool {
        const unsigned int pos = (unsigned)tile * kWideTokens + my_row;
        // a list entry of all ones is nobody's token, and only the 8-bit modes count it (as attend_part)
        const bool nobody = MODE != kDense && tok == 0xffffffffu && !a.count_ones;
        const FewRow r = few_row(a, (pos < (unsigned)(r_end - r_begin)) & !nobody, tok, page);
        if (a.bad_rows && hg == 0 && __builtin_amdgcn_ballot_w64(r.bad) != 0) {
            if (r.bad && l8 == 0) atomicAdd(a.bad_rows, 1u);
        }
        few_dma4(r.scale, scalar((lds_ptr<uint8_t>)scale_raw[buf][wave]));
        few_dma_row(r.codes + 16 * (l8 ^ swap), scalar(rows + buf * kWideTileBytes + wave * 4096),
                    scalar(rows + buf * kWideTileBytes + kWideRopeAt + (wave >> 1) * 1024), roped);
        return r.there;
    };

    // ---- prologue: the query is asked for, two tiles are looked up and requested, the lookups of the third made; then
    // the query becomes operands: each wave has its quarter of the 32 heads' dims (two waves the same one).
    const int th = wave & 1, kq = wave >> 1;  // the wave's 32 tokens of a tile's scores, and its quarter of the dims
    const int head = hg * kWideHeads + n32;
    // First of K-step j's eight dims of the lane's half. Two K-steps share a 16-byte piece of codes.
    auto dim_of = [&](int j) -> int { return j == 8 ? kKvl + 16 * kq + 8 * half : 128 * kq + 32 * (j >> 1) + 16 * half + 8 * (j & 1); };
    float4 qv[kWideSteps][2];
    {
        const size_t qrow = (size_t)seq * a.H + (head < a.H ? head : 0);
#pragma unroll
        for (int j = 0; j < kWideSteps; ++j) {
            const float* src = j < 8 ? a.qabs + qrow * kKvl + dim_of(j) : a.qrope + qrow * kRopeW + (dim_of(j) - kKvl);
            qv[j][0] = reinterpret_cast<const float4*>(src)[0], qv[j][1] = reinterpret_cast<const float4*>(src)[1];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    bool there0 = false, there1 = false;  // the lane's row of this tile, and of the next
    {
        const unsigned int tok0 = token_of(0, my_row), tok1 = token_of(1, my_row);
        const unsigned int tok2 = token_of(2, 8 * wave + l8), tok3 = token_of(3, 8 * wave + l8);
        const int page0 = *entry_of(tok0), page1 = *entry_of(tok1);
        const int page2 = *entry_of(tok2);
        if (lane < 8) {
            token_smem[2][wave][lane] = tok2, token_smem[3][wave][lane] = tok3;
            page_smem[2][wave][lane] = page2;
        }
        __builtin_amdgcn_sched_barrier(0);
        there0 = request(0, 0, tok0, page0);
        if (n_tiles > 1) there1 = request(1, 1, tok1, page1);
    }
    bf16x8 qh[kWideSteps], ql[QSPLIT == 2 ? kWideSteps : 1];
    {
        const float keep = head < a.H ? a.qscale : 0.0f;
#pragma unroll
        for (int j = 0; j < kWideSteps; ++j) {
            const float v[8] = {qv[j][0].x, qv[j][0].y, qv[j][0].z, qv[j][0].w, qv[j][1].x, qv[j][1].y, qv[j][1].z, qv[j][1].w};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float x = v[i] * keep;
                qh[j][i] = (__bf16)x;
                if (QSPLIT == 2) ql[j][i] = (__bf16)(x - (float)qh[j][i]);
            }
        }
    }

    // O^T: the wave's columns in two tiles of 32, sixteen of them a lane, of head n32
    f32x16 o[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) o[c] = f32x16{};
    // The softmax's: four tokens of one head a lane, four heads a wave.
    const int own = 4 * wave + (lane >> 4), four = 4 * (lane & 15);
    float m_ref = -INFINITY, l_sum = 0.0f;

    // The lane's operands of a tile. Scores: row 32 th + n32, pieces 2 i + half of the quarter's group. Values: of sixteen lanes, pair e
    // addresses row 8 (half) + e of sixteen tokens; column tile c is pieces 2 (wave & 1) + c of group wave >> 1 and, in the other sixteen lanes, 4
    // further on, which keeps the two in different banks.
    const int k_swap = (n32 >> 1) & 7, e8 = (lane & 15) >> 1;
    const int k_row = (4 * th + (n32 >> 3)) * 4096 + 1024 * kq + (n32 & 7) * 128;
    const int k_rope = kWideRopeAt + (2 * th + (n32 >> 4)) * 1024 + (n32 & 7) * 128 + 16 * (kq ^ k_swap) + 8 * half;
    const int v_swap = 4 * half + (e8 >> 1);
    const int v_row = half * 4096 + (wave >> 1) * 1024 + e8 * 128 + 8 * (lane & 1);
    const int v_piece = 2 * (wave & 1) + 4 * ((lane >> 4) & 1);
    const lds_ptr<uint8_t> p_at = weights + n32 * (2 * kWideTokens);
    const int p_swap = (n32 >> 1) & 7;
    auto as_bf16 = [](uint32_t x, uint32_t y) -> bf16x8 {
        uint32_t d0, d1, d2, d3;
        e4m3x4_to_bf16(x, d0, d1), e4m3x4_to_bf16(y, d2, d3);
        const u32x4 d = {d0, d1, d2, d3};
        return __builtin_bit_cast(bf16x8, d);
    };

    // The tile's transfers have landed (`more`: all but the last ones, the next tile's): its missing rows and its scales.
    auto arrived = [&](int tile, int buf, bool there, bool more) {
        if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kWideInFlight) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (__builtin_amdgcn_ballot_w64(!there) != 0 && !there) {  // codes must be finite, they meet a zero weight
            const lds_ptr<uint8_t> to = rows + buf * kWideTileBytes + 16 * lane;
#pragma unroll
            for (int i = 0; i < 4; ++i) *(lds_ptr<u32x4>)(to + wave * 4096 + 1024 * i) = u32x4{0, 0, 0, 0};
            if (16 * (l8 ^ swap) < kRopeW) *(lds_ptr<u32x4>)(to + kWideRopeAt + (wave >> 1) * 1024) = u32x4{0, 0, 0, 0};
        }
        // a scale that is not a positive number cannot come from the append: such a token is
        // left out like one that is not there
        const float x = scale_raw[buf][wave][lane];
        if (l8 == 0) scale_smem[tile & 1][my_row] = there && x > 0.0f ? x : 0.0f;
    };
    bf16x8 f[4][2];  // the values' operands of the tile before
    // O^T[column][head] += V^T . P^T
    auto values = [&]() {
        const float corr = corr_smem[n32];
        bf16x8 p[4], p_lo[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const lds_ptr<uint8_t> at = p_at + 16 * ((2 * ks + half) ^ p_swap);
            p[ks] = *(lds_ptr<bf16x8>)at;
            if (PSPLIT == 2) p_lo[ks] = *(lds_ptr<bf16x8>)(at + kWideHeads * kWideTokens * 2);
        }
        if (__builtin_amdgcn_ballot_w64(corr != 1.0f) != 0) {
#pragma unroll
            for (int c = 0; c < 2; ++c) o[c] *= corr;
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int u = 0; u < PSPLIT; ++u)
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[ks][c], u ? p_lo[ks] : p[ks], o[c], 0, 0, 0);
    };

    if (n_tiles > 0) arrived(0, 0, there0, n_tiles > 1);
    __syncthreads();
    int buf = 0;
    for (int tile = 0; tile < n_tiles; ++tile) {
        const lds_ptr<uint8_t> codes = rows + buf * kWideTileBytes;
        // ---- this tile's scores: S^T[token][head] of the wave's 32 tokens over its quarter of the dims; the next tile but one
        // is requested, into the buffer of the tile before; and that tile's values.
        u32x4 k[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) k[i] = *(lds_ptr<u32x4>)(codes + k_row + 16 * ((2 * i + half) ^ k_swap));
        const u32x2 rope = *(lds_ptr<u32x2>)(codes + k_rope);
        bool there2 = false;
        if (tile + 2 < n_tiles) {
            const int t2 = (tile + 2) & 3, t3 = (tile + 3) & 3, t4 = tile & 3;
            const unsigned int tok = rows_g ? token_smem[t2][wave][lane >> 3] : at_of(tile + 2, my_row);
            const int page = page_smem[t2][wave][lane >> 3];
            const unsigned int tok3 = rows_g ? token_smem[t3][wave][l8] : at_of(tile + 3, 8 * wave + l8);
            if (lane < 8) few_dma4(entry_of(tok3), scalar((lds_ptr<uint8_t>)page_smem[t3][wave]));
            if (rows_g && lane < 8) few_dma4(rows_g + at_of(tile + 4, 8 * wave + l8), scalar((lds_ptr<uint8_t>)token_smem[t4][wave]));
            there2 = request(tile + 2, buf == 0 ? 2 : buf - 1, tok, page);
        }
        if (tile > 0) values();
        {
            f32x16 s = {}, s_lo = {};
            auto step = [&](int j, bf16x8 x) {
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, qh[j], s, 0, 0, 0);
                if (QSPLIT == 2) s_lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, ql[j], s_lo, 0, 0, 0);
            };
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                step(2 * i, as_bf16(k[i].x, k[i].y));
                step(2 * i + 1, as_bf16(k[i].z, k[i].w));
            }
            step(8, as_bf16(rope.x, rope.y));
            if (QSPLIT == 2) s += s_lo;
            const lds_ptr<float> to = scores + (kWideHeads * kq + n32) * kWideScoreStride + 32 * th + 4 * half;
#pragma unroll
            for (int i = 0; i < 4; ++i) *(lds_ptr<f32x4>)(to + 8 * i) = f32x4{s[4 * i], s[4 * i + 1], s[4 * i + 2], s[4 * i + 3]};
        }
        __syncthreads();

        // ---- online softmax, each score once, while the values' operands come out of LDS: the transposing
        // load hands a lane the codes of one column for its eight tokens
        i32x2 raw[4][2];
        {
            f32x4 part[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) part[i] = *(lds_ptr<f32x4>)(scores + (kWideHeads * i + own) * kWideScoreStride + four);
            const f32x4 scl = *(lds_ptr<f32x4>)((lds_ptr<float>)scale_smem[tile & 1] + four);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const lds_ptr<uint8_t> at = codes + v_row + 16 * ((v_piece + c) ^ v_swap);
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) raw[ks][c] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr<i32x2>)(at + 8192 * ks));
            }
            float x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = scl[i] > 0.0f ? ((part[0][i] + part[1][i]) + (part[2][i] + part[3][i])) * scl[i] : -INFINITY;
            float tmax = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
            tmax = few_max16(tmax);
            const bool grow = tmax > m_ref + kLazyRescale;  // false while nothing is there
            const float corr = grow ? __builtin_amdgcn_exp2f(m_ref - tmax) : 1.0f;  // 2^-inf = 0 at first
            if (grow) m_ref = tmax;
            if ((lane & 15) == 0) corr_smem[own] = corr;
            l_sum *= corr;
            const float mu = m_ref == -INFINITY ? 0.0f : m_ref;
            // the weights under their tokens' scales
            typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
            bf16x4 hi, lo;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float e = __builtin_amdgcn_exp2f(x[i] - mu);  // not there -> 0
                const float y = e * scl[i];
                hi[i] = (__bf16)y;
                if (PSPLIT == 2) {
                    lo[i] = (__bf16)(y - (float)hi[i]);
                    l_sum += e;
                } else {
                    l_sum += (float)hi[i] * (scl[i] > 0.0f ? __builtin_amdgcn_rcpf(scl[i]) : 0.0f);
                }
            }
            const lds_ptr<uint8_t> to = weights + own * (2 * kWideTokens) + 16 * ((four >> 3) ^ ((own >> 1) & 7)) + 2 * (four & 7);
            *(lds_ptr<bf16x4>)to = hi;
            if (PSPLIT == 2) *(lds_ptr<bf16x4>)(to + kWideHeads * kWideTokens * 2) = lo;
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int c = 0; c < 2; ++c) f[ks][c] = as_bf16((uint32_t)raw[ks][c][0], (uint32_t)raw[ks][c][1]);
        buf = buf == 2 ? 0 : buf + 1;
        if (tile + 1 < n_tiles) arrived(tile + 1, buf, there1, tile + 2 < n_tiles);
        there1 = there2;
        __syncthreads();
    }
    if (n_tiles > 0) values();

    // ---- results: of column tile c a lane's registers 4 i .. are dims of piece 2 (wave & 1) + c, or 4 pieces further on (i >= 2),
    // from 8 (i & 1) + 4 half on
    l_sum += few_dpp<0x128>(l_sum), l_sum += few_dpp<0x124>(l_sum), l_sum += few_dpp<0x122>(l_sum), l_sum += few_dpp<0x121>(l_sum);
    if ((lane & 15) == 0) ml_smem[own][0] = m_ref, ml_smem[own][1] = l_sum;
    __syncthreads();
    if (head < a.H) {
        const float m = ml_smem[n32][0], l = ml_smem[n32][1];
        float* const dst = (whole ? a.clat + (size_t)seq * a.H * kKvl : pa) + (size_t)head * kKvl + 128 * (wave >> 1) + 32 * (wave & 1) + 4 * half;
        const float fin = !whole ? 1.0f : l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<f32x4*>(dst + 16 * c + 64 * (i >> 1) + 8 * (i & 1)) =
                    f32x4{o[c][4 * i] * fin, o[c][4 * i + 1] * fin, o[c][4 * i + 2] * fin, o[c][4 * i + 3] * fin};
        if (!whole && wave == 0 && half == 0) pml[head * 2] = m, pml[head * 2 + 1] = l;
    }
}

}  // namespace rk
