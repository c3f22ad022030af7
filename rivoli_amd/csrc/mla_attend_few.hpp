// MLA decode attention by workgroups of 16 heads, eight waves on one 64-token tile: the same arithmetic, work
// items and records as mla_attend_heads16.hpp (bf16 matrix instructions, q and the weights as bf16 hi + lo in
// the parity mode), which a call takes being a rule of mla_attend_plan.hpp (heads16_few). Included by mla_attend.hip.
//
// A short call is a chain: list entry, table, row, scores, softmax, values, merge. A tile of its own per wave has
// 128 tokens in work in a workgroup, so 33 rows keep two of its four waves and every call pays for the merge of four
// waves' 16 x 512 accumulators through LDS. Here all eight waves (two per SIMD, so that one issues while
// the other waits) share a tile: a wave brings in eight of its rows, has 16 tokens' scores over half of the dims, two heads'
// softmax (two tokens a lane: an exponential is computed once) and 64 columns of the values, whose accumulators are
// final. Scores and weights pass through LDS; two barriers a tile, one before the softmax of the tile and one after it:
// the section between them has the values' operands come out of LDS under it, the other one has this tile's scores and the values
// of the tile before.
// Codes stay codes in LDS (a tile is 40 KB, three of them: this one, the next, and the next but one on its way) and become bf16 when
// an operand is read, twice in all for a workgroup; a form that staged bf16 through registers was bound by its
// LDS writes (43.2 us where this one takes 36.2, the first of the calls below).
// Every read from memory in the loop is a transfer into LDS, list entries, pages and scales too: a load into a register
// would have the compiler wait for it, and with it for the rows that were asked for before it.
// Measured, parity mode, with the merge of the records: 64 heads, 6 ragged sequences of up to 9 000 tokens 39.2 -> 36.2 us
// (with the append), 8 x 2 048 listed rows 24 -> 20; linear slabs, 2 048 rows 19.2 -> 17.0, 300 rows 19.4 -> 13.7, 33 rows 12.6 -> 7.1. Of a
// tile's cycles 1 090 a wave are matrix instructions. Since, by a lookup without branches, a row's transfers by one address, lane maxima of an
// instruction a step and the cut found without lane shuffles: the first 35.7 -> 33.2, the listed rows' launch 16.9 -> 15.8, the linear slabs' 12.6 -> 11.5.
#pragma once

namespace rk {

constexpr int kFewWaves = 8;
constexpr int kFewThreads = kFewWaves * kWave;
constexpr int kFewTokens = 64;                       // of a tile
constexpr int kFewColTiles = kKvl / 16 / kFewWaves;  // a wave's column tiles
constexpr int kFewSteps = kKSteps / 2;               // a wave's K-steps of 32 dims: half of a row's
constexpr int kFewBuffers = 3;
// A tile in LDS: 5 KB of each wave, its eight rows in five groups of 128 bytes (the codes, then the roped keys), a group's
// rows next to each other. A row's eight 16-byte pieces of a group change places by the row's number, so that sixteen
// rows' reads of one piece, and those of its neighbour by other lanes, meet in no bank.
constexpr int kFewWaveBytes = 5 * 1024;
constexpr int kFewTileBytes = kFewWaves * kFewWaveBytes;
constexpr int kFewScoreStride = kFewTokens + 4;
constexpr int kFewInFlight = 6;                      // a tile's transfers by a wave, after its lookups
static_assert(kKSteps == 18 && kRowW == 576 && kKSteps * 2048 <= kFewTileBytes, "the query's operands pass through a buffer");

template <int CTRL>
__device__ __forceinline__ float few_dpp(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}
// max over sixteen lanes, in each of them: an instruction a step (the compiler's maximum quiets both operands first, and takes a move for
// the other lane's). The wait before each is what a lane's value needs on its way to another.
__device__ __forceinline__ float few_max16(float x) {
    asm("s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf"
        : "+v"(x));
    return x;
}
// max / sum over 32 lanes, in each of them
__device__ __forceinline__ float few_max32(float x) {
    x = few_max16(x);
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float few_sum32(float x) {
    x += few_dpp<0x128>(x), x += few_dpp<0x124>(x), x += few_dpp<0x122>(x), x += few_dpp<0x121>(x);
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
// Four bytes per lane from memory into LDS, as dma16.
__device__ __forceinline__ void few_dma4(const void* src, lds_ptr<uint8_t> dst) {
    const uint32_t base = (uint32_t)(uintptr_t)dst;
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(src), "s"(base)
                 : "memory");
}

// A lane's four pieces of a row's codes, 128 bytes apart in memory and 1024 in LDS, and its fifth, of the roped codes, for the lanes of
// `roped`. The instruction's offset counts in memory and in LDS, so m0 makes up the difference and the address is one. All lanes are here.
__device__ __forceinline__ void few_dma_row(const uint8_t* src, lds_ptr<uint8_t> to, lds_ptr<uint8_t> to_rope, unsigned long long roped) {
    const uint32_t base = (uint32_t)(uintptr_t)to, rope = (uint32_t)(uintptr_t)to_rope - 512u;
    uint32_t keep;
    unsigned long long all;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\t"
                 "s_add_u32 m0, m0, 896\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off offset:128\n\t"
                 "s_add_u32 m0, m0, 896\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off offset:256\n\t"
                 "s_add_u32 m0, m0, 896\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off offset:384\n\t"
                 "s_mov_b32 m0, %4\n\ts_and_saveexec_b64 %1, %5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off offset:512\n\t"
                 "s_mov_b64 exec, %1\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep), "=&s"(all)
                 : "v"(src), "s"(base), "s"(rope), "s"(roped)
                 : "memory", "scc");
}

// A paged row, looked up: whether it is there, its codes and its scale (of one that is not there the first row's). bad: it should be.
struct FewRow {
    bool there, bad;
    const uint8_t *codes, *scale;
};
__device__ __forceinline__ FewRow few_row(const AttendArgs& a, bool mine, unsigned int tok, int page) {
    unsigned int blk, off;
    if (a.page_shift >= 0) blk = tok >> a.page_shift, off = tok & (unsigned)(a.page_tokens - 1);
    else blk = tok / (unsigned)a.page_tokens, off = tok - blk * (unsigned)a.page_tokens;
    FewRow r;
    r.there = mine & (blk < (unsigned)a.max_blocks) & ((unsigned)page < (unsigned)a.n_pages);
    r.bad = mine & !r.there;
    off = r.there ? off : 0u;
    const uint8_t* const base = a.pool + (unsigned long long)(unsigned)(r.there ? page : 0) * a.page_bytes;
    r.codes = base + (unsigned long long)off * (unsigned)kRowW;
    r.scale = base + (size_t)a.page_tokens * kRowW + (unsigned long long)off * 4u;
    return r;
}

// One part of a workgroup's work, as attend_part: rows [r_begin, r_end) of sequence `seq`, heads
// 16 * hg .. +15.
template <int QSPLIT, int PSPLIT, int MODE>
__device__ __forceinline__ void attend_part_few(const AttendArgs& a, int seq, int hg, int r_begin, int r_end,
                                                bool whole, float* pa, float* pml) {
    constexpr bool LINEAR = MODE == kLinear;
    static_assert(!LINEAR || (QSPLIT == 2 && PSPLIT == 2), "the linear slabs run in the parity mode");
    constexpr int kScales = LINEAR ? 4 : 1;         // a token's
    __shared__ __attribute__((aligned(1024))) uint8_t smem[kFewBuffers * kFewTileBytes];
    __shared__ __attribute__((aligned(16))) float score_smem[2 * kH16Heads * kFewScoreStride];
    __shared__ __attribute__((aligned(16))) uint8_t weight_smem[kScales * PSPLIT * kH16Heads * kFewTokens * 2];
    __shared__ __attribute__((aligned(16))) float scale_smem[2][kScales][kFewTokens];  // by the tile's parity
    __shared__ __attribute__((aligned(16))) float there_smem[2][LINEAR ? kFewTokens : 4];
    __shared__ __attribute__((aligned(16))) float scale_raw[kFewBuffers][kFewWaves][kWave];
    // a tile's list entries and pages, 8 a wave, by the tile's number
    __shared__ __attribute__((aligned(16))) unsigned int token_smem[4][kFewWaves][8];
    __shared__ __attribute__((aligned(16))) int page_smem[4][kFewWaves][8];
    __shared__ float corr_smem[kH16Heads], ml_smem[kH16Heads][2];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, n16 = lane & 15;
    const int n_tiles = (r_end - r_begin + kFewTokens - 1) / kFewTokens;
    const lds_ptr<uint8_t> rows = (lds_ptr<uint8_t>)smem;
    const lds_ptr<float> scores = (lds_ptr<float>)score_smem;
    const lds_ptr<uint8_t> weights = (lds_ptr<uint8_t>)weight_smem;

    // ---- where a tile's rows are: eight lanes ask for row 8 wave + (lane >> 3) ---------------------------------
    const int my_row = 8 * wave + (lane >> 3), l8 = lane & 7;
    const unsigned int* const rows_g = MODE == kSparse ? a.rows + (size_t)seq * a.k : (LINEAR ? a.rows : nullptr);
    const int* const table_g = LINEAR ? nullptr : a.block_table + (size_t)seq * a.max_blocks;
    // a row's place in the list (or its position), clamped: lookups run past the end
    // (unsigned: tiles past the end of 2^31 - 32 rows are past what an int holds)
    auto at_of = [&](int tile, int row) -> unsigned int {
        return min((unsigned)r_begin + (unsigned)tile * kFewTokens + (unsigned)row, (unsigned)r_end - 1u);
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
        const unsigned int pos = (unsigned)tile * kFewTokens + my_row;
        // a list entry of all ones is nobody's token, and only the 8-bit modes count it (as attend_part)
        const bool nobody = MODE != kDense && tok == 0xffffffffu && (LINEAR || !a.count_ones);
        const bool mine = (pos < (unsigned)(r_end - r_begin)) & !nobody;
        const int piece = 16 * (l8 ^ swap);
        const lds_ptr<uint8_t> to = scalar(rows + buf * kFewTileBytes + wave * kFewWaveBytes);
        const lds_ptr<uint8_t> to_scale = scalar((lds_ptr<uint8_t>)scale_raw[buf][wave]);
        if constexpr (LINEAR) {  // a row that is not there reads the first one
            const size_t t = mine ? tok : 0;
            few_dma4(reinterpret_cast<const uint8_t*>(a.lscale + t * 4 + (l8 & 3)), to_scale);
#pragma unroll
            for (int i = 0; i < 4; ++i) dma16(a.lc8 + t * kKvl + piece + 128 * i, to + 1024 * i);
            dma16(reinterpret_cast<const uint8_t*>(a.rc + t * kRopeW) + piece, to + 4096);
            return mine;
        } else {
            const FewRow r = few_row(a, mine, tok, page);
            if (a.bad_rows && hg == 0 && __builtin_amdgcn_ballot_w64(r.bad) != 0) {
                if (r.bad && l8 == 0) atomicAdd(a.bad_rows, 1u);
            }
            few_dma4(r.scale, to_scale);
            few_dma_row(r.codes + piece, to, to + 4096, roped);
            return r.there;
        }
    };

    // ---- prologue: the query is asked for, two tiles are looked up and requested, the lookups of the third made; then
    // each wave turns every eighth K-step of the 16 heads into operands, and takes its own half of them.
    const int head = hg * kH16Heads + n16;
    // First of K-step j's eight dims of lane group g. Two K-steps share a 16-byte piece of codes; the linear slabs' roped keys
    // are bf16, eight a piece.
    auto dim_of = [&](int j) -> int {
        if (j >= 16) return kKvl + (LINEAR ? 32 * (j - 16) + 8 * g : 16 * g + 8 * (j - 16));
        return 64 * (j >> 1) + 16 * g + 8 * (j & 1);
    };
    constexpr int kMine = (kKSteps + kFewWaves - 1) / kFewWaves;
    float4 qv[kMine][2];
    {
        const size_t qrow = (size_t)seq * a.H + (head < a.H ? head : 0);
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            const int d = dim_of(min(wave + m * kFewWaves, kKSteps - 1));
            const float* src = d < kKvl ? a.qabs + qrow * kKvl + d : a.qrope + qrow * kRopeW + (d - kKvl);
            qv[m][0] = reinterpret_cast<const float4*>(src)[0], qv[m][1] = reinterpret_cast<const float4*>(src)[1];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    bool there0 = false, there1 = false;  // the lane's row of this tile, and of the next
    {
        const unsigned int tok0 = token_of(0, my_row), tok1 = token_of(1, my_row);
        const unsigned int tok2 = token_of(2, 8 * wave + l8), tok3 = token_of(3, 8 * wave + l8);
        const int page0 = LINEAR ? 0 : *entry_of(tok0), page1 = LINEAR ? 0 : *entry_of(tok1);
        const int page2 = LINEAR ? 0 : *entry_of(tok2);
        if (lane < 8) {
            token_smem[2][wave][lane] = tok2, token_smem[3][wave][lane] = tok3;
            if (!LINEAR) page_smem[2][wave][lane] = page2;
        }
        __builtin_amdgcn_sched_barrier(0);
        there0 = request(0, 0, tok0, page0);
        if (n_tiles > 1) there1 = request(1, 1, tok1, page1);
    }
    const lds_ptr<uint8_t> q_room = rows + 2 * kFewTileBytes + 16 * lane;
    {
        const float keep = head < a.H ? a.qscale : 0.0f;
#pragma unroll
        for (int m = 0; m < kMine; ++m) {
            const int j = wave + m * kFewWaves;
            if (j >= kKSteps) break;  // wave-uniform
            const float v[8] = {qv[m][0].x, qv[m][0].y, qv[m][0].z, qv[m][0].w, qv[m][1].x, qv[m][1].y, qv[m][1].z, qv[m][1].w};
            bf16x8 hi, lo;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float x = v[i] * keep;
                hi[i] = (__bf16)x;
                lo[i] = (__bf16)(x - (float)hi[i]);
            }
            *(lds_ptr<bf16x8>)(q_room + j * 2048) = hi;
            if (QSPLIT == 2) *(lds_ptr<bf16x8>)(q_room + j * 2048 + 1024) = lo;
        }
    }
    __syncthreads();
    const int tg = wave & 3, kh = wave >> 2;  // the wave's 16 tokens of a tile's scores, and its half of the dims
    bf16x8 qh[kFewSteps], ql[QSPLIT == 2 ? kFewSteps : 1];
#pragma unroll
    for (int i = 0; i < kFewSteps; ++i) {
        const int j = i < 8 ? 8 * kh + i : 16 + kh;
        qh[i] = *(lds_ptr<bf16x8>)(q_room + j * 2048);
        if (QSPLIT == 2) ql[i] = *(lds_ptr<bf16x8>)(q_room + j * 2048 + 1024);
    }

    // O^T: columns 16-tile c of the wave's 64, four of them a lane, of head n16
    f32x4 o[kFewColTiles];
#pragma unroll
    for (int c = 0; c < kFewColTiles; ++c) o[c] = f32x4{0, 0, 0, 0};
    // The softmax's: two tokens of one head a lane, two heads a wave.
    const int own = 2 * wave + (lane >> 5), pair = 2 * (lane & 31);
    float m_ref = -INFINITY, l_sum = 0.0f;

    // the lane's operands of a tile: row 16 tg + n16 of the scores, pieces 4 i + g of the wave's half; rows 8 g + (n16 >> 1)
    // (and 32 further on) of the values
    const int k_swap = n16 >> 1, v_swap = (4 * (g & 1) + (n16 >> 2)) & 7;
    const int k_row = (2 * tg + (n16 >> 3)) * kFewWaveBytes + (n16 & 7) * 128;
    const int k_even = k_row + 2048 * kh + 16 * (g ^ k_swap), k_odd = k_row + 2048 * kh + 16 * ((4 + g) ^ k_swap);
    const int k_rope = k_row + 4096 + (LINEAR ? 16 * ((4 * kh + g) ^ k_swap) : 16 * (g ^ k_swap) + 8 * kh);
    const int v_row = g * kFewWaveBytes + (n16 >> 1) * 128 + (wave >> 1) * 1024 + 8 * (n16 & 1);
    auto as_bf16 = [](uint32_t x, uint32_t y) -> bf16x8 {
        uint32_t d0, d1, d2, d3;
        e4m3x4_to_bf16(x, d0, d1), e4m3x4_to_bf16(y, d2, d3);
        const u32x4 d = {d0, d1, d2, d3};
        return __builtin_bit_cast(bf16x8, d);
    };

    // The tile's transfers have landed (`more`: all but the last ones, the next tile's): its missing rows and its scales.
    auto arrived = [&](int tile, int buf, bool there, bool more) {
        if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFewInFlight) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (__builtin_amdgcn_ballot_w64(!there) != 0 && !there) {  // codes must be finite, they meet a zero weight
            const lds_ptr<uint8_t> to = rows + buf * kFewTileBytes + wave * kFewWaveBytes + 16 * lane;
#pragma unroll
            for (int i = 0; i < 5; ++i) *(lds_ptr<u32x4>)(to + 1024 * i) = u32x4{0, 0, 0, 0};
        }
        // a scale that is not a positive number cannot come from the append: such a token is
        // left out like one that is not there (linear slabs: a token is there or it is not)
        const float x = scale_raw[buf][wave][lane];
        const lds_ptr<float> scl = (lds_ptr<float>)scale_smem[tile & 1][0];
        if constexpr (LINEAR) {
            if (l8 < 4) scl[l8 * kFewTokens + my_row] = there ? x : 0.0f;
            if (l8 == 0) there_smem[tile & 1][my_row] = there ? 1.0f : 0.0f;
        } else {
            if (l8 == 0) scl[my_row] = there && x > 0.0f ? x : 0.0f;
        }
    };
    bf16x8 f[2][kFewColTiles];  // the values' operands of the tile before
    // O^T[column][head] += V^T . P^T
    auto values = [&](float corr, const bf16x8 (&p)[2], const bf16x8 (&p_lo)[2]) {
        if (__builtin_amdgcn_ballot_w64(corr != 1.0f) != 0) {
#pragma unroll
            for (int c = 0; c < kFewColTiles; ++c) o[c] *= corr;
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int u = 0; u < PSPLIT; ++u)
#pragma unroll
                for (int c = 0; c < kFewColTiles; ++c)
                    o[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[ks][c], u ? p_lo[ks] : p[ks], o[c], 0, 0, 0);
    };
    auto take_weights = [&](float& corr, bf16x8 (&p)[2], bf16x8 (&p_lo)[2]) {
        corr = corr_smem[n16];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const lds_ptr<uint8_t> at = weights + (LINEAR ? (wave >> 1) * PSPLIT * 2048 : 0) + n16 * 128 + 16 * ((4 * ks + g) ^ (n16 >> 1));
            p[ks] = *(lds_ptr<bf16x8>)at;
            if (PSPLIT == 2) p_lo[ks] = *(lds_ptr<bf16x8>)(at + 2048);
        }
    };

    if (n_tiles > 0) arrived(0, 0, there0, n_tiles > 1);
    __syncthreads();
    int buf = 0;
    for (int tile = 0; tile < n_tiles; ++tile) {
        const lds_ptr<uint8_t> codes = rows + buf * kFewTileBytes;
        const lds_ptr<float> scl = (lds_ptr<float>)scale_smem[tile & 1][0];
        // ---- this tile's scores: S^T[token][head] of the wave's 16 tokens over its half of the dims; the next tile but one
        // is requested, into the buffer of the tile before; and that tile's values.
        f32x4 s = {0, 0, 0, 0}, s_lo = {0, 0, 0, 0}, t = {0, 0, 0, 0};
        f32x4 sb[2];
        u32x4 k[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) k[i] = *(lds_ptr<u32x4>)(codes + ((i & 1) ? k_odd : k_even) + 1024 * (i >> 1));
        bf16x8 rope;
        u32x2 rope_code;
        if constexpr (LINEAR) {
            rope = *(lds_ptr<bf16x8>)(codes + k_rope);
#pragma unroll
            for (int b = 0; b < 2; ++b) sb[b] = *(lds_ptr<f32x4>)(scl + (2 * kh + b) * kFewTokens + 16 * tg + 4 * g);
        } else {
            rope_code = *(lds_ptr<u32x2>)(codes + k_rope);
        }
        float corr;
        bf16x8 p[2], p_lo[2];
        if (tile > 0) take_weights(corr, p, p_lo);
        bool there2 = false;
        if (tile + 2 < n_tiles) {
            const int t2 = (tile + 2) & 3, t3 = (tile + 3) & 3, t4 = tile & 3;
            const unsigned int tok = rows_g ? token_smem[t2][wave][lane >> 3] : at_of(tile + 2, my_row);
            int page = 0;
            if constexpr (!LINEAR) {
                page = page_smem[t2][wave][lane >> 3];
                const unsigned int tok3 = rows_g ? token_smem[t3][wave][l8] : at_of(tile + 3, 8 * wave + l8);
                if (lane < 8) few_dma4(entry_of(tok3), scalar((lds_ptr<uint8_t>)page_smem[t3][wave]));
            }
            if (rows_g && lane < 8) few_dma4(rows_g + at_of(tile + 4, 8 * wave + l8), scalar((lds_ptr<uint8_t>)token_smem[t4][wave]));
            there2 = request(tile + 2, buf == 0 ? 2 : buf - 1, tok, page);
        }
        if (tile > 0) values(corr, p, p_lo);
        {
            auto step = [&](int i, bf16x8 f) {
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, qh[i], s, 0, 0, 0);
                if (QSPLIT == 2) s_lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, ql[i], s_lo, 0, 0, 0);
            };
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                step(2 * i, as_bf16(k[i].x, k[i].y));
                step(2 * i + 1, as_bf16(k[i].z, k[i].w));
                if (LINEAR && (i & 1)) {  // the block's dots under its scales
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[e] += (s[e] + s_lo[e]) * sb[i >> 1][e];
                    s = s_lo = f32x4{0, 0, 0, 0};
                }
            }
            if constexpr (!LINEAR) rope = as_bf16(rope_code.x, rope_code.y);
            step(8, rope);
            if (QSPLIT == 2) s += s_lo;
            if (LINEAR) s += t;
            *(lds_ptr<f32x4>)(scores + (16 * kh + n16) * kFewScoreStride + 16 * tg + 4 * g) = s;
        }
        __syncthreads();

        // ---- online softmax, each score once, while the values' operands come out of LDS, all of the wave's: the transposing
        // load hands a lane the codes of one column for its eight tokens; source lane pair e addresses token e's row
        i32x2 raw[2][kFewColTiles];
        {
            typedef float f32x2 __attribute__((ext_vector_type(2)));
            const f32x2 v = *(lds_ptr<f32x2>)(scores + own * kFewScoreStride + pair), w = *(lds_ptr<f32x2>)(scores + (16 + own) * kFewScoreStride + pair);
            const f32x2 is = LINEAR ? *(lds_ptr<f32x2>)((lds_ptr<float>)there_smem[tile & 1] + pair) : *(lds_ptr<f32x2>)(scl + pair);
#pragma unroll
            for (int c = 0; c < kFewColTiles; ++c) {
                const lds_ptr<uint8_t> at = codes + v_row + 16 * ((4 * (wave & 1) + c) ^ v_swap);
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) raw[ks][c] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr<i32x2>)(at + 4 * kFewWaveBytes * ks));
            }
            float x[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) x[i] = is[i] > 0.0f ? (v[i] + w[i]) * (LINEAR ? 1.0f : is[i]) : -INFINITY;
            const float tmax = few_max32(fmaxf(x[0], x[1]));
            const bool grow = tmax > m_ref + kLazyRescale;  // false while nothing is there
            const float corr = grow ? __builtin_amdgcn_exp2f(m_ref - tmax) : 1.0f;  // 2^-inf = 0 at first
            if (grow) m_ref = tmax;
            if ((lane & 31) == 0) corr_smem[own] = corr;
            l_sum *= corr;
            const float mu = m_ref == -INFINITY ? 0.0f : m_ref;
            const float e[2] = {__builtin_amdgcn_exp2f(x[0] - mu), __builtin_amdgcn_exp2f(x[1] - mu)};  // not there -> 0
            // the weights under their tokens' scales (linear slabs: those of each column block)
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            const lds_ptr<uint8_t> to = weights + own * 128 + 16 * ((pair >> 3) ^ ((own >> 1) & 7)) + 2 * (pair & 7);
#pragma unroll
            for (int b = 0; b < kScales; ++b) {
                const f32x2 sc = LINEAR ? *(lds_ptr<f32x2>)(scl + b * kFewTokens + pair) : is;
                bf16x2 hi, lo;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float y = e[i] * sc[i];
                    hi[i] = (__bf16)y;
                    if (PSPLIT == 2) {
                        lo[i] = (__bf16)(y - (float)hi[i]);
                        if (b == 0) l_sum += e[i];
                    } else {
                        l_sum += (float)hi[i] * (sc[i] > 0.0f ? __builtin_amdgcn_rcpf(sc[i]) : 0.0f);
                    }
                }
                *(lds_ptr<bf16x2>)(to + b * PSPLIT * 2048) = hi;
                if (PSPLIT == 2) *(lds_ptr<bf16x2>)(to + b * PSPLIT * 2048 + 2048) = lo;
            }
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int c = 0; c < kFewColTiles; ++c) f[ks][c] = as_bf16((uint32_t)raw[ks][c][0], (uint32_t)raw[ks][c][1]);
        buf = buf == 2 ? 0 : buf + 1;
        if (tile + 1 < n_tiles) arrived(tile + 1, buf, there1, tile + 2 < n_tiles);
        there1 = there2;
        __syncthreads();
    }
    if (n_tiles > 0) {
        float corr;
        bf16x8 p[2], p_lo[2];
        take_weights(corr, p, p_lo);
        values(corr, p, p_lo);
    }

    // ---- results: a lane's four columns of tile c are dims 64 wave + 16 c + 4 g ..
    l_sum = few_sum32(l_sum);
    if ((lane & 31) == 0) ml_smem[own][0] = m_ref, ml_smem[own][1] = l_sum;
    __syncthreads();
    if (head < a.H) {
        const float m = ml_smem[n16][0], l = ml_smem[n16][1];
        float* const dst = (whole ? a.clat + (size_t)seq * a.H * kKvl : pa) + (size_t)head * kKvl + 64 * wave + 4 * g;
        const float fin = !whole ? 1.0f : l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
        for (int c = 0; c < kFewColTiles; ++c) *reinterpret_cast<f32x4*>(dst + 16 * c) = o[c] * fin;
        if (!whole && wave == 0 && g == 0) pml[head * 2] = m, pml[head * 2 + 1] = l;
    }
}

}  // namespace rk
