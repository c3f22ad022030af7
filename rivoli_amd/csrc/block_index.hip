// The second cache format's block indexer: the Hadamard + simulated-fp4 spread of its q rows
// and of its compressor's pooled rows, and the block scorer that ranks compressed blocks for a
// query (crates/backend/kernels/blockindex.hip:99-136 and :209-235, launchers :241-281; CPU
// statements crates/oracles/src/v4oracle/numerics.rs:245-353 and
// crates/engine/tests/kernel_v4_indexer.rs:437-462). Both are bit-exact by construction: every
// value is produced by the reference's tree of f32 operations; what differs is who computes
// which value and where the operands wait.
//
// Spread. The reference gives a row to a 128-thread workgroup and walks LDS log2(d) times with
// a barrier per stage, then hands each fp4 block of 32 to one thread. Here a lane holds four
// consecutive values of a row (one 16-byte load and store, a wave moves 1 KiB per instruction),
// d / 4 neighbouring lanes hold a row, and a wave holds 64 / (d / 4) rows. The butterflies of
// stages 1 and 2 pair values of one lane; stage h >= 4 pairs lane L with lane L ^ (h / 4): the
// lane whose bit is clear holds the pair's first value and computes a + b, the other computes
// a - b from the same two numbers. A block of 32 is eight lanes; its amax is a maximum (exact
// in any order) over three lane exchanges. No LDS, no barrier; 8 bytes of traffic per value.
//
// Scorer. score[t][c] = bf16(sum_h bf16(relu(bf16(q[t][h] . kv[c])) * w[t][h])), the dot a
// sequential f32 fold of separately rounded products and the head sum a sequential f32 fold
// (blockindex.hip:138-207 argues each). In general that order rules out the matrix cores and
// any split of a dot over lanes. But the rows the indexer hands over are spread rows: a handful
// of significant bits each, over a few binades. Every product and every partial sum of two such
// rows is a multiple of one power of two and fits 24 bits, so no addition rounds and EVERY order
// gives the reference's bits. The matrix kernels (hd = 128, up to 64 heads) test that property
// on the operands they hold (RowSpan) and take such tiles through v_mfma_f32_32x32x16_bf16; any
// other tile of the same launch is folded term by term as below; rows that are fp4 codes under
// powers of two, as spread rows are, go through the block-scaled fp4 instruction. 8 192 queries x 64 heads x
// <= 2 048 blocks: 160 us, 226 as bf16, 3 640 term by term.
// Operands of another kind (no such rows leave the indexer) take the same launches' fold: 3 430.
// Term by term, what is free is where the operands come from. A lane owns block c and
// keeps its 128-value row in registers for the whole launch; a wave's 64 lanes share the query,
// so q[t][h][i] and w[t][h] are wave-uniform and come through scalar loads straight into the
// multiply's scalar operand. Per (t, h) a wave issues 128 multiplies and 128 adds for 64
// scores and reads 512 bytes through the scalar cache: bound by vector issue, two
// instructions per multiply-add because the reference's rounding is two roundings.
// Widths other than 128 re-read the block's row through the vector cache instead.
#include "block_index_plan.hpp"
#include "codec.hpp"

#include <cmath>
#include <type_traits>

#include "rivoli_kvcache.h"

#pragma clang fp contract(off)

namespace rk {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float kFp4Max = 6.0f;
constexpr float kFp4MaxInv = 1.0f / kFp4Max;
constexpr float kFp4AmaxFloor = kFp4Max * 1.17549435082228750797e-38f;  // 6 * 2^-126 (actquant.hpp:51)
constexpr int kSpreadMaxD = 256;   // blockindex.hip:40-42
constexpr int kSpreadThreads = 256;
// Row groups per wave, all requested before the first is used: 4, or 1 where that leaves fewer
// workgroups than compute units (a wave's row groups are worked on one after the other: 64 rows of
// 128, a decode step's, 5.0 -> 3.0 us; one row 3.4 -> 1.8).
constexpr int kSpreadInFlight = 4;
constexpr int kSpreadFewGroups = 256;

// bf16(x) as a float: the conversion of the pair (0, x) leaves it in the upper half, one instruction.
__device__ __forceinline__ float round_bf16(float x) {
    return __builtin_bit_cast(float, __builtin_convertvector(f32x2{0.0f, x}, bf16x2));
}

// formats.hpp:285-293 followed by its decode, for |q| <= 6: the nearest of {0, .5, 1, 1.5, 2, 3,
// 4, 6}, a tie to the even mantissa. The grid is spaced .5 below 2, 1 below 4 and 2 above, and
// on each stretch "tie to the even mantissa" is "tie to the even multiple of the spacing"
// (.25 -> 0, .75 -> 1, 1.25 -> 1, 1.75 -> 2, 2.5 -> 2, 3.5 -> 4, 5 -> 4: the reference's own
// table), which is what adding and subtracting 2^22, 2^23 or 2^24 does in round-to-nearest-even
// f32 arithmetic: two compares and two additions where counting midpoints takes fourteen
// instructions. A NaN passes no midpoint there and becomes a zero with its sign; here too.
__device__ __forceinline__ float e2m1_round_trip(float q) {
    const float a = fabsf(q);
    const float magic = a < 2.0f ? 4194304.0f : (a < 4.0f ? 8388608.0f : 16777216.0f);
    float v = (a + magic) - magic;
    v = a != a ? 0.0f : v;
    return __builtin_signbit(q) ? -v : v;
}

// LPR: lanes per row (d / 4). scale = 1 / sqrt(d), taken on the host (a correctly rounded
// square root and a true divide, blockindex.hip:107-113).
template <int LPR, int IN_FLIGHT>
__global__ __launch_bounds__(kSpreadThreads) void f4_rotated_kernel(float* __restrict__ x,
                                                                     long long rows, float scale) {
    constexpr int kRowsPerWave = kWave / LPR;
    constexpr int d = LPR * 4;
    const int lane = threadIdx.x & (kWave - 1);
    const long long wave = (long long)blockIdx.x * (kSpreadThreads / kWave) + (threadIdx.x >> 6);
    const long long row0 = wave * (kRowsPerWave * IN_FLIGHT) + lane / LPR;
    const int col = (lane % LPR) * 4;

    f32x4 v[IN_FLIGHT];
#pragma unroll
    for (int u = 0; u < IN_FLIGHT; ++u) {
        const long long r = row0 + (long long)u * kRowsPerWave;
        // unconditional: a row past the end re-reads the last row and is not stored
        v[u] = *reinterpret_cast<const f32x4*>(x + (r < rows ? r : rows - 1) * d + col);
    }
#pragma unroll
    for (int u = 0; u < IN_FLIGHT; ++u) {
        float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
        // stages h = 1, 2: inside the lane
        {
            const float a0 = e[0] + e[1], a1 = e[0] - e[1], a2 = e[2] + e[3], a3 = e[2] - e[3];
            e[0] = a0 + a2, e[2] = a0 - a2, e[1] = a1 + a3, e[3] = a1 - a3;
        }
        // stages h = 4 .. d / 2: lane L with lane L ^ (h / 4)
#pragma unroll
        for (int m = 1; m < LPR; m <<= 1) {
            const bool upper = (lane & m) != 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float other = __shfl_xor(e[i], m, kWave);
                e[i] = upper ? other - e[i] : e[i] + other;
            }
        }
        // the bf16 store between rotation and quantization (blockindex.hip:91-96)
        float amax = kFp4AmaxFloor;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            e[i] = round_bf16(e[i] * scale);
            amax = fmaxf(amax, fabsf(e[i]));
        }
        // a block of 32 is 8 lanes; d = 32 is the whole row
#pragma unroll
        for (int m = 1; m < 8; m <<= 1) amax = fmaxf(amax, __shfl_xor(amax, m, kWave));
        // actquant.hpp:65-75: the smallest power of two >= amax / 6, by exponent surgery
        const uint32_t b = __float_as_uint(amax * kFp4MaxInv);
        const int ex = (int)((b >> 23) & 0xffu) - 127 + ((b & 0x7fffffu) ? 1 : 0);
        const float s = __uint_as_float((uint32_t)(ex + 127) << 23);
        // x / s for a power of two s is x * (1 / s) exactly whenever 1 / s is a normal number
        // (one multiply instead of the divide's dozen instructions); the divide stays for the
        // scales at the ends of the exponent range
        const bool by_reciprocal = ex >= -126 && ex <= 126;
        const float rinv = __uint_as_float((uint32_t)(127 - ex) << 23);
        f32x4 out;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float q = by_reciprocal ? e[i] * rinv : e[i] / s;
            q = q < -kFp4Max ? -kFp4Max : (q > kFp4Max ? kFp4Max : q);  // a NaN stays a NaN
            out[i] = round_bf16(e2m1_round_trip(q) * s);
        }
        const long long r = row0 + (long long)u * kRowsPerWave;
        if (r < rows) *reinterpret_cast<f32x4*>(x + r * d + col) = out;
    }
}

// ---- the block scorer -------------------------------------------------------------------------
constexpr int kScoreThreads = 256;           // four waves, 64 blocks each
constexpr int kScoreQueriesPerGroup = 16;    // queries a workgroup walks with its rows held

// The scalar operands of one 32-term chunk of a dot. Scalar loads return out of order, so the
// only wait there is waits for all of them: a chunk is requested one whole chunk of
// arithmetic (64 vector instructions) before it is used and nothing else is outstanding then.
struct QChunk {
    float v[32];
};
__device__ __forceinline__ void load_chunk(QChunk& c, const float* __restrict__ p) {
#pragma unroll
    for (int i = 0; i < 32; ++i) c.v[i] = p[i];
}
// Waits for the chunk here: placed before the next chunk is requested, the wait covers this
// chunk alone (requested a chunk ago); left to the first use it would also cover the request
// just made.
__device__ __forceinline__ void arrived(const QChunk& c) {
    asm volatile("" ::"s"(c.v[0]), "s"(c.v[16]));
}
template <int OFF>
__device__ __forceinline__ float fold_chunk(float dot, const QChunk& c, const float (&row)[128]) {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const float prod = c.v[i] * row[OFF + i];
        dot = dot + prod;
    }
    return dot;
}

// bf16 first, then the relu (blockindex.hip:224-228; the sign of a zero cannot reach the
// output), the weight, the term's own bf16 store, the f32 head sum.
__device__ __forceinline__ float head_term(float dot, float weight) {
    dot = round_bf16(dot);
    dot = dot > 0.0f ? dot : 0.0f;
    const float term = dot * weight;
    return round_bf16(term);
}

// Which (query group, block group) a workgroup owns. The full rectangle runs block groups
// fastest (ratio == 0): the workgroups that share a query group start together, one per die,
// and their q rows are fetched from memory once for all of them (7.0 ms against 7.4 at 8 192 x
// 2 048). The prefill form runs query groups fastest: workgroups are dealt to the 8 dies in
// turn, and with block groups fastest (often 8 of them) each die would own one block group,
// whose work shrinks with its index — the first die would do an eighth of the rectangle alone
// while the last one idles (6.8 ms against 3.4).
__device__ __forceinline__ int query_group(int ratio) { return ratio > 0 ? blockIdx.x : blockIdx.y; }
__device__ __forceinline__ int block_group(int ratio) { return ratio > 0 ? blockIdx.y : blockIdx.x; }

// The first of the workgroup's queries [t0, t1) this wave scores. ratio > 0 is a prefill whose
// selection ranks block c for query t only when c < (t + 1) / ratio (a block is legal once it
// has closed): a wave's 64 blocks start at cw, and no query before ratio * (cw + 1) - 1 can
// rank any of them.
__device__ __forceinline__ int first_query(int t0, int t1, int ratio, long long cw) {
    if (ratio <= 0) return t0;
    const long long first = (cw + 1) * ratio - 1;
    return first > t0 ? (int)(first < t1 ? first : t1) : t0;
}

// The lane's block row, 128 values, into registers.
__device__ __forceinline__ void load_row(float (&row)[128], const float* __restrict__ kvr) {
#pragma unroll
    for (int i = 0; i < 128; i += 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(kvr + i);
        row[i] = v.x, row[i + 1] = v.y, row[i + 2] = v.z, row[i + 3] = v.w;
    }
}

// One head term, bf16(relu(bf16(q . row)) * weight), for each (query, head) pair g in [g0, g1):
// the pairs' 128-value q rows are contiguous and are walked as one run through two chunk
// buffers. on_term(g, term) receives them in order.
template <class OnTerm>
__device__ __forceinline__ void walk_pairs(const float* __restrict__ q, const float* __restrict__ w,
                                           const float (&row)[128], size_t g0, size_t g1,
                                           OnTerm&& on_term) {
    constexpr int HD = 128;
    if (g0 >= g1) return;  // (wave-uniform) no pair: the first chunk below would be pair g1's
    const float* qp = q + g0 * HD;
    QChunk a, b;
    load_chunk(a, qp);
    for (size_t g = g0; g < g1; ++g) {
        float dot = 0.0f;
        arrived(a);
        const float weight = w[g];
        load_chunk(b, qp + 32);
        __builtin_amdgcn_sched_barrier(0);
        dot = fold_chunk<0>(dot, a, row);
        __builtin_amdgcn_sched_barrier(0);
        arrived(b);
        load_chunk(a, qp + 64);
        __builtin_amdgcn_sched_barrier(0);
        dot = fold_chunk<32>(dot, b, row);
        __builtin_amdgcn_sched_barrier(0);
        arrived(a);
        load_chunk(b, qp + 96);
        __builtin_amdgcn_sched_barrier(0);
        dot = fold_chunk<64>(dot, a, row);
        __builtin_amdgcn_sched_barrier(0);
        arrived(b);
        load_chunk(a, g + 1 < g1 ? qp + HD : qp);  // the next pair's first chunk; the last re-reads its own
        __builtin_amdgcn_sched_barrier(0);
        dot = fold_chunk<96>(dot, b, row);
        __builtin_amdgcn_sched_barrier(0);
        on_term(g, head_term(dot, weight));
        qp += HD;
    }
}

// hd = 128 past the matrix kernels' 64 heads, many (query, block group) pairs: a lane owns a block for the workgroup's queries
// and folds the head terms itself, in head order.
__global__ __launch_bounds__(kScoreThreads) void index_score_blocks_128_kernel(
    const float* __restrict__ q, const float* __restrict__ kv, const float* __restrict__ w,
    float* __restrict__ score, int s, int n_comp, int heads, int t_per_group, int ratio) {
    const long long c = (long long)block_group(ratio) * kScoreThreads + threadIdx.x;
    const int t1 = min(s, query_group(ratio) * t_per_group + t_per_group);
    const long long cw = (long long)block_group(ratio) * kScoreThreads +
                         (__builtin_amdgcn_readfirstlane((int)threadIdx.x) & ~(kWave - 1));
    const int t0 = first_query(query_group(ratio) * t_per_group, t1, ratio, cw);
    if (t0 >= t1) return;  // wave-uniform; the kernel has no barrier
    float row[128];
    load_row(row, kv + (size_t)(c < n_comp ? c : n_comp - 1) * 128);
    float acc = 0.0f;
    int hh = 0, t = t0;
    walk_pairs(q, w, row, (size_t)t0 * heads, (size_t)t1 * heads, [&](size_t, float term) {
        acc = acc + term;
        if (++hh == heads) {
            if (c < n_comp) score[(size_t)t * n_comp + c] = round_bf16(acc);
            acc = 0.0f, hh = 0, ++t;
        }
    });
}

// hd = 128, 65 to 128 heads, few (query, block group) pairs (a decode step: one query): the plain kernel would
// occupy n_comp / 256 compute units for 64 heads' worth of arithmetic each. Here a workgroup
// owns 64 blocks and its eight waves each take an eighth of the heads: the dots of different
// heads are independent, only their sum has an order. The head terms meet in LDS and the first
// wave folds them in head order, as the reference does.
constexpr int kSplitWavesPerGroup = 8;
constexpr int kSplitMaxHeads = 128;  // 32 KiB of terms
__global__ __launch_bounds__(kSplitWavesPerGroup* kWave) void index_score_blocks_128_split_kernel(
    const float* __restrict__ q, const float* __restrict__ kv, const float* __restrict__ w,
    float* __restrict__ score, int s, int n_comp, int heads, int ratio) {
    extern __shared__ float terms[];  // [heads][64]
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const long long cw = (long long)blockIdx.x * kWave;
    const long long c = cw + lane;
    const int t0 = first_query(0, s, ratio, cw);  // the same for every wave: the barriers below are safe
    const int per = (heads + kSplitWavesPerGroup - 1) / kSplitWavesPerGroup;
    const int h0 = min(wave * per, heads), h1 = min(h0 + per, heads);
    float row[128];
    load_row(row, kv + (size_t)(c < n_comp ? c : n_comp - 1) * 128);
    for (int t = t0; t < s; ++t) {
        const size_t base = (size_t)t * heads;
        walk_pairs(q, w, row, base + h0, base + h1,
                   [&](size_t g, float term) { terms[(g - base) * kWave + lane] = term; });
        __syncthreads();
        if (wave == 0) {
            float acc = 0.0f;
            for (int hh = 0; hh < heads; ++hh) acc = acc + terms[hh * kWave + lane];
            if (c < n_comp) score[(size_t)t * n_comp + c] = round_bf16(acc);
        }
        __syncthreads();
    }
}

// ---- the matrix kernels -------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef f32x4 f32x4_u __attribute__((aligned(4)));  // q rows need no more than a float's alignment

// When is q . kv the same in every order? Let the non-zero values of a row have exponents in
// [lo, hi] and at most two significant bits (1 or 1.5 times a power of two: what e2m1 times a
// power of two is). Its values are multiples of 2^(lo - 1) and at most 1.5 * 2^hi. A sum of up to
// 128 products of two rows is then a multiple of u = 2^(lo_q + lo_kv - 2) below 288 * 2^(hi_q +
// hi_kv), that is below 2^(10.2 + (hi_q - lo_q) + (hi_kv - lo_kv)) u: with (hi_q - lo_q) + (hi_kv -
// lo_kv) <= 13 every partial sum is a whole number of u below 2^24 and every f32 addition is
// exact. Exponents within +-59 keep u a normal number and every sum below 288 * 2^118 < 2^127 (at
// 60 a fold may pass the largest float where another order does not). A spread row spans 3
// binades plus what its four block scales differ by; 13 leaves 7 for those.
constexpr int kExactSpan = 13;
constexpr int kNoSpan = 99;  // not such a row: no partner makes it exact
// The census of a row, two bf16 patterns per dword: largest magnitude in the low 16 bits' field,
// 0xffff - (smallest non-zero magnitude - 1) in the high one, so both fold by a packed maximum.
struct RowSpan {
    u16x2 hi = {0, 0}, lo = {0xffff, 0xffff};
    uint32_t low_bits = 0;
    // p: two bf16 patterns; bits: the OR of the low mantissa halves of the f32 values they came from
    __device__ __forceinline__ void add(uint32_t p, uint32_t bits) {
        low_bits |= bits | (p & 0x003f003fu);
        const u16x2 m = __builtin_bit_cast(u16x2, p & 0x7fff7fffu);
        hi = __builtin_elementwise_max(hi, m);
        lo = __builtin_elementwise_min(lo, (u16x2)(m - (u16x2){1, 1}));  // a zero wraps to 0xffff
    }
    __device__ __forceinline__ uint32_t folded() const {
        const uint32_t h = hi.x > hi.y ? hi.x : hi.y, l = lo.x < lo.y ? lo.x : lo.y;
        return low_bits ? 0xffffffffu : (h | ((0xffffu - l) << 16));
    }
};
__device__ __forceinline__ uint32_t span_max(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a),
                                                                  __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ int span_of(uint32_t folded) {
    const int hi = (int)((folded & 0xffffu) >> 7), lo = (int)((0x10000u - (folded >> 16)) >> 7);
    if (!(folded & 0xffffu)) return 0;  // a row of zeros
    return hi > 127 + 59 || lo < 127 - 59 ? kNoSpan : hi - lo;
}
// Two f32 bit patterns to a dword of two bf16 patterns by truncation (exact when the census finds
// no low bits).
__device__ __forceinline__ uint32_t upper_halves(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ uint32_t low_half_bits(const f32x4& v) {
    return (__float_as_uint(v.x) | __float_as_uint(v.y) | __float_as_uint(v.z) | __float_as_uint(v.w)) & 0xffffu;
}

// The fold of rows that are not exact in every order. Scalar operands (walk_pairs) want waves that
// share their q rows and three of them a SIMD; the matrix kernels' fold has neither, and waited for
// the scalar cache a quarter of its time. Here every sixteen lanes hold a q row in eight registers,
// lane j of them dims 4 j + e and 64 + 4 j + e, and a multiply takes dim i from lane (i % 64) / 4 of
// its own sixteen (row_newbcast: an operand modifier, no instruction). Vector loads return in order,
// so a row is requested a whole dot (256 instructions) before it is used, and the halves of a wave may
// fold different rows. f32 values of no particular kind, 64 heads, prefill form, us: folded by
// scalar operands in kernels of their own (walk_pairs) / by them in the matrix kernels / so:
// 8 192 x 2 048 3 640 / 4 800 / 3 430, 4 096 x 1 024 1 050 / 1 290 / 970, 2 000 x 500 282 / 472 / 422,
// 1 000 x 250 83 / 157 / 120, 300 x 75 39 / 88 / 44; the full form, 5 x 8 192 39 / 83 / 44, 1 x 8 192 14 /
// 18 / 13. Not reached: 2 x 16 384 21 / 78 / 73 and 1 x 16 384 14 / 18.6 / 18.6, whose eight waves a
// workgroup shared the heads, and 5 heads, 8 192 x 2 048 256 / 431 / 507, where fetching a row outweighs it.
struct QRow {
    f32x4 v[2];
};
__device__ __forceinline__ QRow load_q(const float* __restrict__ at) {  // at: the row + 4 * (lane & 15)
    return {{*reinterpret_cast<const f32x4_u*>(at), *reinterpret_cast<const f32x4_u*>(at + 64)}};
}
template <int I>
__device__ __forceinline__ float q_dim(const QRow& q) {
    constexpr int kRowNewBcast = 0x150;  // | lane of the sixteen
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(q.v[I / 64][I % 4]), kRowNewBcast | (I % 64) / 4, 0xf, 0xf, true));
}
// Every addition needs the one before it, so the next dim's product is taken between two of them.
// SHARED: another wave is on the SIMD. Two waves without a pause take 4.6 cycles an instruction
// between them, with an empty slot after each addition 4.0; a wave alone 5.0, and 6.8 with the slot.
template <bool SHARED, int I = 0>
__device__ __forceinline__ float fold_dot(float dot, float prod, const QRow& q, const float (&row)[128]) {
    if constexpr (I == 127) {
        return dot + prod;
    } else {
        const float next = q_dim<I + 1>(q) * row[I + 1];
        __builtin_amdgcn_sched_barrier(0);
        dot = dot + prod;
        __builtin_amdgcn_sched_barrier(0);
        if (SHARED) asm volatile("s_nop 0");
        return fold_dot<SHARED, I + 1>(dot, next, q, row);
    }
}
// The head terms of `n` >= 1 consecutive heads from the lane's first on, whose q row and weight are at
// q and w. on_term(i, term) receives them in order. All lanes of the wave must be here.
template <bool SHARED, class OnTerm>
__device__ __forceinline__ void fold_heads(const float* __restrict__ q, const float* __restrict__ w, int n,
                                           const float (&row)[128], OnTerm&& on_term) {
    q += 4 * (threadIdx.x & 15);
    QRow next = load_q(q);
    float next_w = *w;
    for (int i = 0; i < n; ++i) {
        const QRow now = next;
        const float weight = next_w;
        if (i + 1 < n) q += 128, ++w;  // the last re-reads its own
        next = load_q(q);
        next_w = *w;
        __builtin_amdgcn_sched_barrier(0);
        on_term(i, head_term(fold_dot<SHARED>(0.0f, q_dim<0>(now) * row[0], now, row), weight));
    }
}

// A workgroup's four waves own two queries each and walk the split's blocks in tiles of 32, which
// all four read from LDS; a wave's q rows stay in registers as matrix operands. The 32 rows of a
// matrix tile are 16 heads of the wave's first query and the same 16 of its second, dealt so that a
// lane's sixteen results are sixteen heads of ONE query in order (the result layout gives lanes 0-31
// the rows with bit 2 clear): the head sum, whose order the reference fixes, is then register arithmetic.
// Bound by issue. As bf16 a lane's 64 dots were 32 matrix instructions of 32 cycles and five vector instructions each (round,
// relu, weight, round, sum); as fp4 codes they are 8 of 32 cycles, and clamping conversions leave four a dot, in steps of which
// none waits for another. 8 192 queries: 226 -> 160 us, of them 120 vector issue (two thirds of it those four; the kv rows' codes, made by every workgroup,
// and the q rows' take the rest), 16 the matrix cores and about 25 the first workgroups' q rows, all asked for at once; 4 096 82 -> 73,
// 6 001 127 -> 102. Not kept: 16 queries a workgroup (half of the conversions; all of q at once, 231), two or three sets of q loads
// in flight (178).
constexpr int kPairWaves = 4;
constexpr int kPairThreads = kPairWaves * kWave;
static_assert(kPairQueries == kPairWaves * 2, "a wave's two queries");
constexpr int kPairHeads = 64;
constexpr int kPairRow = 128 * 2 + 16;  // bytes of a bf16 row in LDS: 16-byte reads of 16 rows meet no bank twice

// Spread rows are what the block-scaled fp4 instruction takes: e2m1 codes, a power of two for 32 of them. A row
// qualifies when every block's values are exactly that (fp4_of); with the block's exponent taken
// from its largest value, products of two rows are multiples of u = 2^(lo_q + lo_kv - 2) and 128 of them sum to
// 128 * 36 * 2^(hi_q + hi_kv) at most, hi and lo being a row's largest and smallest block exponents: below 2^24 u for (hi_q - lo_q) +
// (hi_kv - lo_kv) <= 9, and the instruction keeps 24 bits of a sum (checked at every such difference, with cancelling
// and one-signed sums in either half of K: exact up to 11, 12 being the first at which sums pass 2^24 u far enough to lose a bit).
// The e4m3 form loses bits sooner. A real row's blocks differ by one binade or two.
constexpr int kFp4Span = 9;
constexpr int kFp4Row = 64 + 16;   // bytes of an fp4 row in LDS
constexpr int kFp4MinExp = 127 - 59, kFp4MaxExp = 127 + 59;  // of a row's largest block, as kExactSpan's
// The least exponent that a block's scale is made for. Blocks below it are out of every range above and below here; and a subnormal value, whose
// exponent field is a zero's, is no code under that scale: it cannot pass for a zero, whether the conversions flush it or not.
constexpr int kFp4LeastExp = 32;
// The dots come out scaled, the largest that 128 products can be to just below one, so that the conversion to bf16 clamps to [0,
// 1] and is the relu too; scores are scaled back. Powers of two change no rounding while nothing leaves the normal numbers:
// with weights in 2^+-50, a query's heads within 20 binades (a scaled dot is 2^-44 then, or zero) and scales back of 2^-20 to 2^40,
// terms are at least 2^-114 scaled or not, and bf16 terms' sums are multiples of 2^-121.
constexpr int kFp4Down = 13;       // 128 * 36 < 2^13
constexpr int kFp4Heads = 20, kFp4Back0 = -20, kFp4Back1 = 40;
constexpr uint32_t kFp4Weight0 = 127 - 50, kFp4Weight1 = 127 + 50;
static_assert(kFp4LeastExp > 5 && kFp4MinExp - kFp4LeastExp >= kFp4Heads && kFp4Heads >= kFp4Span, "no block below kFp4LeastExp is taken");

template <int CTRL>
__device__ __forceinline__ uint32_t max_with_lane(uint32_t x) {
    return max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xf, 0xf, true));
}
// Four values of a block that eight neighbouring lanes hold, as fp4 codes under the block's scale. expo: the biased exponent of
// the block's largest magnitude (the scale is 2^(expo - 129): that value becomes 4 or 6), 0 for zeros; off: non-zero when
// a value is not exactly its code.
__device__ __forceinline__ uint32_t fp4_of(const f32x4& v, uint32_t& expo, uint32_t& off) {
    // (assembly: the compiler's maximum quiets each operand first, an instruction more for each)
    float top;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(top) : "v"(v.x), "v"(v.y), "v"(v.z));
    asm("v_max_f32_e64 %0, %1, |%2|" : "=v"(top) : "v"(top), "v"(v.w));
    uint32_t m = __float_as_uint(top);
    m = max_with_lane<0xB1>(m);   // lane ^ 1
    m = max_with_lane<0x4E>(m);   // lane ^ 2
    m = max_with_lane<0x141>(m);  // lane 7 - i: the other four's
    expo = m >> 23;
    const float scale = __uint_as_float((max(expo, (uint32_t)kFp4LeastExp) - 2u) << 23);
    uint32_t c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, v.x, v.y, scale, 0);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, v.z, v.w, scale, 1);
    const f32x2 lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, scale, 0), hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, scale, 1);
    off |= (__float_as_uint(v.x) ^ __float_as_uint(lo.x)) | (__float_as_uint(v.y) ^ __float_as_uint(lo.y));
    off |= (__float_as_uint(v.z) ^ __float_as_uint(hi.x)) | (__float_as_uint(v.w) ^ __float_as_uint(hi.y));
    return c;
}
__device__ __forceinline__ f32x16 fp4_products(const u32x4& a, const u32x4& b, const f32x16& d, int a_scale, int b_scale) {
    typedef int i32x8 __attribute__((ext_vector_type(8)));
    const i32x8 x = {(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0}, y = {(int)b.x, (int)b.y, (int)b.z, (int)b.w, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, y, d, 4, 4, 0, a_scale, 0, b_scale);
}
// f(0), f(1), .. f(N - 1), each a constant.
template <int N, int I = 0, class F>
__device__ __forceinline__ void each_of(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        each_of<N, I + 1>(f);
    }
}
// bf16(relu(x)), and the same for an x of at most one in magnitude. The second is assembly, for which the compiler keeps no distance from a
// matrix instruction: of such an instruction's results it may read those that come out of an empty assembly with a result of the first.
__device__ __forceinline__ float relu_bf16(float x) {
    x = round_bf16(x);
    return x > 0.0f ? x : 0.0f;
}
__device__ __forceinline__ float clamp_bf16(float x) {
    float r;
    asm("v_cvt_pk_bf16_f32 %0, 0, %1 clamp" : "=v"(r) : "v"(x));
    return r;
}

struct PairArgs {
    const float *q, *kv, *w;
    float* score;
    int s, n_comp, heads, split_blocks, ratio;
};
template <bool FP4>
struct PairShared {
    // q rows on their way to operands (a wave's 32 at a time), and kv rows
    __align__(16) unsigned char stage[kPairWaves * 32 * kPairRow];
    __align__(16) float weights[kPairWaves][2][kPairHeads];
    int kv_spans[2][FP4 ? 2 * kPairTile : kPairTile];
    uint32_t row_expo[FP4 ? kPairWaves * 32 : 1], kv_expo[FP4 ? 4 * kPairTile : 1];  // four block exponents a row
    unsigned long long left[kPairWaves][2];
    int fits[kPairWaves];
};
// Tiles from block c0 on of 64-block groups with a block that some query up to t_last may rank (first_query).
__device__ __forceinline__ int pair_tiles(const PairArgs& a, int c0, int t_last) {
    int end = min(a.n_comp, c0 + a.split_blocks);
    if (a.ratio > 0) end = min(end, ((t_last + 1) / a.ratio + 63) & ~63);
    return end > c0 ? (end - c0 + kPairTile - 1) / kPairTile : 0;
}
// Blocks of query t from here on are nobody's: it does not exist, or its selection ranks none of their 64.
__device__ __forceinline__ int pair_limit(const PairArgs& a, int t) {
    return t >= a.s ? 0 : a.ratio <= 0 ? a.n_comp : min(a.n_comp, ((t + 1) / a.ratio + 63) & ~63);
}
struct PairPlace {
    int lane, half, row, wave, kr, kp;  // kv tiles: eight threads (kp) a row (kr), 16-byte pieces
    int tw, t, c0;                      // the wave's first query, the lane's; the workgroup's first block
    int tiles, my_tiles;                // of the workgroup; of the wave
};
__device__ __forceinline__ PairPlace pair_place(const PairArgs& a, int tid) {
    PairPlace at;
    at.lane = tid & (kWave - 1), at.half = at.lane >> 5, at.row = at.lane & 31;
    at.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    at.kr = tid >> 3, at.kp = tid & 7;
    // the last queries of a prefill rank the most blocks: they start first
    const int group = a.ratio > 0 ? (int)gridDim.x - 1 - (int)blockIdx.x : (int)blockIdx.x;
    at.tw = group * kPairQueries + at.wave * 2, at.t = at.tw + at.half;
    at.c0 = blockIdx.y * a.split_blocks;
    at.tiles = pair_tiles(a, at.c0, min(a.s, (group + 1) * kPairQueries) - 1);
    at.my_tiles = at.tw < a.s ? pair_tiles(a, at.c0, min(a.s, at.tw + 2) - 1) : 0;
    return at;
}
// The next kv rows are requested before these ones' products and parked after them.
__device__ __forceinline__ void request_rows(const PairArgs& a, const PairPlace& at, int tile, f32x4 (&to)[4]) {
    const float* const p = a.kv + (size_t)min(at.c0 + tile * kPairTile + at.kr, a.n_comp - 1) * 128 + at.kp * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) to[j] = *reinterpret_cast<const f32x4*>(p + j * 32);
}
// Eight loads of the rows of heads 16 c ..: load m = 2 (j0 + j) + half is row m, head c * 16 + (m >> 3) * 4 + (m & 3) of
// query (m >> 2) & 1; an instruction moves two whole rows.
__device__ __forceinline__ void request_heads(const PairArgs& a, const PairPlace& at, int c, int j0, f32x4 (&v)[8]) {
    const bool all = c * 16 + 16 <= a.heads;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int hh = c * 16 + ((j0 + j) >> 2) * 4 + (2 * (j0 + j) & 3);  // and hh + 1 in the upper half
        const float* const from = a.q + (size_t)min(at.tw + ((j0 + j) >> 1 & 1), a.s - 1) * a.heads * 128;  // uniform
        if (all) v[j] = *reinterpret_cast<const f32x4_u*>(from + hh * 128 + (uint32_t)(at.half * 128 + at.row * 4));
        else v[j] = *reinterpret_cast<const f32x4_u*>(from + (uint32_t)(min(hh + at.half, a.heads - 1) * 128 + at.row * 4));
    }
    __builtin_amdgcn_sched_barrier(0);  // all eight requested before the first is waited for
    if (!all) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (c * 16 + ((j0 + j) >> 2) * 4 + (2 * (j0 + j) & 3) + at.half >= a.heads) v[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
}
// The weights of head `lane`, both queries.
__device__ __forceinline__ void load_weights(const PairArgs& a, const PairPlace& at, float (&x)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) x[i] = at.lane < a.heads ? a.w[(size_t)min(at.tw + i, a.s - 1) * a.heads + at.lane] : 0.0f;
}

// The tiles of `left`, of each wave its own, as bf16 operands where those are exact, the others term by term. ALL: every tile; else sh.left
// holds what each wave has left.
template <bool ALL, class SHARED>
__device__ __forceinline__ void score_left(const PairArgs& a_, const PairPlace& at, SHARED& sh) {
    const int lane = at.lane, half = at.half, row = at.row, wave = at.wave, tw = at.tw, c0 = at.c0, t = at.t, kr = at.kr, kp = at.kp;
    const int tiles = at.tiles, my_tiles = at.my_tiles, s = a_.s, n_comp = a_.n_comp, heads = a_.heads;
    const float* const kv = a_.kv;
    float* const score = a_.score;
    unsigned char* const stage = sh.stage;
    const auto request = [&](int tile, f32x4 (&to)[4]) { request_rows(a_, at, tile, to); };
    const auto load_heads = [&](int c, int j0, f32x4 (&v)[8]) { request_heads(a_, at, c, j0, v); };
    const auto limit_of = [&](int t) { return pair_limit(a_, t); };
    const int limit = limit_of(t);
    auto& weights = sh.weights;
    auto& kv_spans = sh.kv_spans;
    f32x4 next[4];
    unsigned long long left[2] = {0, 0};
    bf16x8 a[4][8];
    int q_span = 0;
    {
        unsigned char* const mine = stage + wave * 32 * kPairRow;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (c * 16 >= heads) break;
            uint32_t low = 0;
#pragma unroll
            for (int j0 = 0; j0 < 16; j0 += 8) {
                f32x4 v[8];
                load_heads(c, j0, v);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    low |= low_half_bits(v[j]);
                    const u32x2 p = {upper_halves(v[j].x, v[j].y), upper_halves(v[j].z, v[j].w)};
                    *reinterpret_cast<u32x2*>(mine + (2 * (j0 + j) + half) * kPairRow + row * 8) = p;
                }
                asm volatile("" ::: "memory");
            }
            if (__any(low != 0)) q_span = kNoSpan;
            asm volatile("" ::: "memory");
            RowSpan span;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const u32x4 p = *reinterpret_cast<const u32x4*>(mine + row * kPairRow + k * 32 + half * 16);
                span.add(p.x, 0), span.add(p.y, 0), span.add(p.z, 0), span.add(p.w, 0);
                a[c][k] = __builtin_bit_cast(bf16x8, p);
            }
            asm volatile("" ::: "memory");
            const uint32_t f = span.folded();
            q_span = max(q_span, span_of(span_max(f, __shfl_xor(f, 32, kWave))));
        }
#pragma unroll
        for (int m = 1; m < 32; m <<= 1) q_span = max(q_span, __shfl_xor(q_span, m, kWave));
    }
    int parity = 0;
    const auto park = [&]() {
        unsigned char* const to = stage + (parity * kPairTile + kr) * kPairRow + kp * 8;
        RowSpan span;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x2 p = {upper_halves(next[j].x, next[j].y), upper_halves(next[j].z, next[j].w)};
            span.add(p.x, low_half_bits(next[j]));
            span.add(p.y, 0);
            *reinterpret_cast<u32x2*>(to + j * 64) = p;
        }
        uint32_t f = span.folded();
        f = span_max(f, __shfl_xor(f, 1, kWave));
        f = span_max(f, __shfl_xor(f, 2, kWave));
        f = span_max(f, __shfl_xor(f, 4, kWave));
        if (kp == 0) kv_spans[parity][kr] = span_of(f);
    };
    if constexpr (ALL) request(0, next);
    __syncthreads();  // every wave's q rows are out of the stage, and its tiles in left_all
    unsigned long long todo[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        todo[k] = 0;
        if constexpr (!ALL) {
            for (int i = 0; i < kPairWaves; ++i) todo[k] |= sh.left[i][k];
            left[k] = sh.left[wave][k];
        } else {
            if (tiles > 64 * k) todo[k] = tiles >= 64 * (k + 1) ? ~0ull : (1ull << (tiles & 63)) - 1;
            if (my_tiles > 64 * k) left[k] = my_tiles >= 64 * (k + 1) ? ~0ull : (1ull << (my_tiles & 63)) - 1;
        }
    }
    const auto pop = [&]() {  // the next of them, or -1
        const int k = todo[0] ? 0 : 1;
        const unsigned long long from = k ? todo[1] : todo[0];
        if (!from) return -1;
        (k ? todo[1] : todo[0]) = from & (from - 1);
        return __builtin_amdgcn_readfirstlane(64 * k + __builtin_ctzll(from));
    };
    unsigned long long inexact[2] = {0, 0};  // one bit per tile
    int tile = pop();
    if constexpr (!ALL) request(tile, next);
    park();
    while (tile >= 0) {
        __syncthreads();
        const int after = pop();
        if (after >= 0) request(after, next);
        if (left[tile >> 6] >> (tile & 63) & 1) {
            if (__any(kv_spans[parity][row] + q_span > kExactSpan)) {
                inexact[tile >> 6] |= 1ull << (tile & 63);
            } else {
                const unsigned char* const from = stage + (parity * kPairTile + row) * kPairRow + half * 16;
                bf16x8 b[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) b[k] = *reinterpret_cast<const bf16x8*>(from + k * 32);
                float acc = 0.0f;
                f32x16 d[2] = {};
#pragma unroll
                for (int k = 0; k < 8; ++k) d[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][k], b[k], d[0], 0, 0, 0);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if (c * 16 >= heads) break;
                    if (c < 3 && (c + 1) * 16 < heads) {
                        f32x16& n = d[(c + 1) & 1];
                        n = f32x16{};
#pragma unroll
                        for (int k = 0; k < 8; ++k) n = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c + 1][k], b[k], n, 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < 16; i += 4) {
                        const f32x4 wv = *reinterpret_cast<const f32x4*>(&weights[wave][half][c * 16 + i]);
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc = acc + head_term(d[c & 1][i + j], wv[j]);
                    }
                }
                const int c = c0 + tile * kPairTile + row;
                if (c < limit)
                    score[(size_t)t * n_comp + c] = round_bf16(acc);
            }
        }
        parity ^= 1;
        if (after >= 0) park();
        tile = after;
    }
    // What is left, term by term: a lane owns a block of a 64-block group for both of the wave's
    // queries, or where only one of the group's tiles is left a block of that for one of them.
    const auto fold = [&](auto shared) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            while (inexact[k]) {
                const int bit = __builtin_ctzll(inexact[k]);
                const bool both = !(bit & 1) && (inexact[k] >> bit & 2);
                inexact[k] &= ~((both ? 3ull : 1ull) << bit);
                const int c = c0 + (64 * k + bit) * kPairTile + (both ? lane : row);
                float row_v[128];
                load_row(row_v, kv + (size_t)min(c, n_comp - 1) * 128);
                const int first = both ? tw : tw + half;
                const size_t from = (size_t)min(first, s - 1) * heads;
                // (both sums first, then the stores: 8 192 x 2 048 3 475 -> 3 425 us)
                float sum = 0.0f, acc = 0.0f;
                fold_heads<shared>(a_.q + from * 128, a_.w + from, both ? min(2, s - tw) * heads : heads, row_v, [&](int i, float term) {
                    acc = acc + term;
                    if (i + 1 == heads) sum = acc, acc = 0.0f;
                });
                if (c < limit_of(first)) score[(size_t)first * n_comp + c] = round_bf16(sum);
                if (both && c < limit_of(tw + 1)) score[(size_t)(tw + 1) * n_comp + c] = round_bf16(acc);
            }
        }
    };
    // (a prefill's grid has a third and more workgroups without a legal block)
    if (gridDim.x * gridDim.y <= (a_.ratio > 0 ? 384u : 256u))
        fold(std::false_type{});
    else
        fold(std::true_type{});
}

__global__ __launch_bounds__(kPairThreads, 2) void score_blocks_pair_kernel(const PairArgs args) {
    __shared__ PairShared<false> sh;
    const PairPlace at = pair_place(args, threadIdx.x);
    if (!at.tiles) return;  // workgroup-uniform
    float own_weights[2];
    load_weights(args, at, own_weights);
#pragma unroll
    for (int i = 0; i < 2; ++i) sh.weights[at.wave][i][at.lane] = own_weights[i];
    score_left<true>(args, at, sh);
}

template <class SHARED>
__device__ __forceinline__ bool score_codes(const PairArgs& a_, const PairPlace& at, SHARED& sh) {
    const int lane = at.lane, half = at.half, row = at.row, wave = at.wave, tw = at.tw, c0 = at.c0, t = at.t, kr = at.kr, kp = at.kp;
    const int tiles = at.tiles, my_tiles = at.my_tiles, s = a_.s, n_comp = a_.n_comp, heads = a_.heads;
    const float* const kv = a_.kv;
    float* const score = a_.score;
    unsigned char* const stage = sh.stage;
    const auto request = [&](int tile, f32x4 (&to)[4]) { request_rows(a_, at, tile, to); };
    const auto load_heads = [&](int c, int j0, f32x4 (&v)[8]) { request_heads(a_, at, c, j0, v); };
    const auto limit_of = [&](int t) { return pair_limit(a_, t); };
    const int limit = limit_of(t);
    auto& weights = sh.weights;
    auto& kv_spans = sh.kv_spans;
    auto& row_expo = sh.row_expo;
    auto& kv_expo = sh.kv_expo;
    auto& wave_fits = sh.fits;
    float own_weights[2];
    load_weights(a_, at, own_weights);
    unsigned long long left[2] = {0, 0};  // one bit per tile that the fp4 products did not do
    f32x4 next[2][4];  // two tiles at a time
    request(0, next[0]);
    request(1, next[1]);  // (past the last block: that one again)
    unsigned char* const kv_codes = stage + kPairWaves * 32 * kFp4Row;
    // Row 32 u + kr of buffer `buf`; whether it is made of codes.
    const auto park = [&](int buf, int u) -> bool {
        const int place = (2 * buf + u) * kPairTile + kr;
        unsigned char* const to = kv_codes + place * kFp4Row + kp * 2;
        uint32_t off = 0, e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<uint16_t*>(to + j * 16) = (uint16_t)fp4_of(next[u][j], e[j], off);
        const uint32_t hi = max(max(e[0], e[1]), max(e[2], e[3]));
        uint32_t lo = min(min(e[0], e[1]), min(e[2], e[3]));
        if (__any(lo == 0)) {  // a block of zeros takes the largest's scale
#pragma unroll
            for (int j = 0; j < 4; ++j) e[j] = e[j] ? e[j] : hi;
            lo = min(min(e[0], e[1]), min(e[2], e[3]));
        }
        // 127 + e - hi in each byte (none of them borrows where the row is taken)
        const uint32_t expo = (e[0] | e[1] << 8 | e[2] << 16 | e[3] << 24) + 0x7f7f7f7fu - __builtin_amdgcn_perm(hi, hi, 0u);
        uint32_t span = hi - lo;
        if (hi - (uint32_t)kFp4MinExp > (uint32_t)(kFp4MaxExp - kFp4MinExp) && hi) span = kNoSpan;
        const unsigned long long bad = __ballot(off != 0);
        if (bad) span = bad >> (lane & ~7) & 0xffu ? (uint32_t)kNoSpan : span;
        // (eight threads, one word)
        kv_expo[place] = expo;
        kv_spans[buf][u * kPairTile + kr] = (int)(span | hi << 8);
        return off == 0;
    };
    bool fits = my_tiles > 0;
    // ---- the rows as fp4 operands: lane's row of a matrix tile, blocks half and 2 + half of its four ----
    u32x4 a[4][2];
    uint32_t a_expo[4] = {};
    unsigned char* const mine = stage + wave * 32 * kFp4Row;
    uint32_t off = 0;
    int top = 0, bottom = 255, apart = 0;  // block exponents: the rows' largest, smallest; largest difference in a row
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c * 16 >= heads || (c == 1 && !fits)) break;
#pragma unroll
        for (int j0 = 0; j0 < 16; j0 += 8) {
            f32x4 v[8];
            load_heads(c, j0, v);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int m = 2 * (j0 + j) + half;
                uint32_t expo;
                *reinterpret_cast<uint16_t*>(mine + m * kFp4Row + row * 2) = (uint16_t)fp4_of(v[j], expo, off);
                // (eight lanes, one byte)
                reinterpret_cast<unsigned char*>(row_expo)[(wave * 32 + m) * 4 + (row >> 3)] = (unsigned char)expo;
            }
            asm volatile("" ::: "memory");  // no more than eight rows' loads in registers at a time
        }
        asm volatile("" ::: "memory");  // the rows cross lanes: LDS serves a wave in order, the compiler must keep to it
#pragma unroll
        for (int k = 0; k < 2; ++k) a[c][k] = *reinterpret_cast<const u32x4*>(mine + row * kFp4Row + (2 * k + half) * 16);
        const uint32_t x = row_expo[wave * 32 + row];
        int hi = 0, lo = 255;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = (int)(x >> (8 * k) & 0xffu);
            hi = max(hi, e), lo = min(lo, e ? e : 255);
        }
        top = max(top, hi), bottom = min(bottom, lo), apart = max(apart, hi - lo);  // a row of zeros: -255
        a_expo[c] = x >> (8 * half);
        asm volatile("" ::: "memory");
        // Where some of the first sixteen heads' values, or of the wave's own rows of the first two tiles, are no codes, hardly any are.
        if (c == 0) {
            const bool codes[2] = {park(0, 0), park(0, 1)};
            if (__any(!codes[0] || !codes[1] || off != 0)) fits = false;
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        weights[wave][i][lane] = own_weights[i];
        const uint32_t e = (__float_as_uint(own_weights[i]) & 0x7fffffffu) >> 23;
        if (own_weights[i] != 0.0f && (e < kFp4Weight0 || e > kFp4Weight1)) off = 1;  // (a NaN differs from zero)
    }
    asm volatile("" ::: "memory");
    if (__any(off != 0)) fits = false;
#pragma unroll
    for (int m = 1; m < 32; m <<= 1) {
        top = max(top, __shfl_xor(top, m, kWave)), bottom = min(bottom, __shfl_xor(bottom, m, kWave));
        apart = max(apart, __shfl_xor(apart, m, kWave));
    }
    top = __builtin_amdgcn_readfirstlane(top), bottom = __builtin_amdgcn_readfirstlane(bottom), apart = __builtin_amdgcn_readfirstlane(apart);
    if (top != 0 && (top > kFp4MaxExp || top < kFp4MinExp || top - bottom > kFp4Heads)) fits = false;
    // scales relative to the largest (a block of zeros takes that)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int e0 = (int)(a_expo[c] & 0xffu), e1 = (int)(a_expo[c] >> 16 & 0xffu);
        a_expo[c] = (uint32_t)(127 - kFp4Down + (e0 ? e0 - top : 0)) | (uint32_t)(127 - kFp4Down + (e1 ? e1 - top : 0)) << 8;
    }
    f32x4 wv[kPairHeads / 4];
#pragma unroll
    for (int i = 0; i < kPairHeads / 4; ++i) wv[i] = *reinterpret_cast<const f32x4*>(&weights[wave][half][4 * i]);

    if (!fits) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (my_tiles > 64 * k) left[k] = my_tiles >= 64 * (k + 1) ? ~0ull : (1ull << (my_tiles & 63)) - 1;
    }
    if (lane == 0) wave_fits[wave] = fits;
    __syncthreads();
    bool some = false;
#pragma unroll
    for (int i = 0; i < kPairWaves; ++i) some = some || wave_fits[i];
    const int walk = some ? tiles : 0;
    for (int tile = 0, buf = 0; tile < walk; tile += 2, buf ^= 1) {
        __syncthreads();  // these tiles are parked and nobody reads the other buffer any more
        if (tile + 2 < tiles) {
            request(tile + 2, next[0]);
            request(tile + 3, next[1]);  // (past the last block: that one again)
        }
        if (fits && tile < my_tiles) {
            u32x4 b[2][2];
            int b_expo[2], info[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int place = (2 * buf + u) * kPairTile + row;
                const unsigned char* const from = kv_codes + place * kFp4Row + half * 16;
                b[u][0] = *reinterpret_cast<const u32x4*>(from), b[u][1] = *reinterpret_cast<const u32x4*>(from + 32);
                b_expo[u] = (int)(kv_expo[place] >> (8 * half));
                info[u] = kv_spans[buf][u * kPairTile + row];
            }
            const auto products = [&](int u, int c) {
                f32x16 d = {};
                d = fp4_products(a[c][0], b[u][0], d, (int)a_expo[c], b_expo[u]);
                return fp4_products(a[c][1], b[u][1], d, (int)(a_expo[c] >> 8), b_expo[u] >> 16);
            };
            f32x16 d = products(0, 0);
            const auto taken = [&](int u) {
                const int back = top + (info[u] >> 8) - 2 * 129 + kFp4Down;  // the scores' scale
                const bool zero = (info[u] >> 8) == 0 || top == 0;
                return !__any(max(apart, 0) + (info[u] & 0xff) > kFp4Span || (!zero && (back < kFp4Back0 || back > kFp4Back1)));
            };
            const bool take[2] = {taken(0), taken(1)};
            float acc = 0.0f;
            const auto finish = [&](int u, int info) {
                const int c = c0 + (tile + u) * kPairTile + row;
                if (c < limit) score[(size_t)t * n_comp + c] = round_bf16(__builtin_amdgcn_ldexpf(acc, top + (info >> 8) - 2 * 129 + kFp4Down));
                acc = 0.0f;
            };
            if (!take[0]) left[tile >> 6] |= 1ull << (tile & 63);
            if (!take[1] && tile + 1 < my_tiles) left[tile >> 6] |= 2ull << (tile & 63);
            if (heads > 48 && take[0] && take[1]) {
                // A step has a head's conversion, the weight of the one before, the rounding of the one before that and the sum's
                // addition of a fourth: four instructions of which none waits for another. The next sixteen
                // heads' products run under these heads' steps. (The sum is finished before the store's branch: used only there, the compiler
                // would put all of its steps there, after the products.)
                constexpr int kSteps = 2 * kPairHeads;
                f32x16 sets[2];
                sets[0] = d;
                float clamped = 0.0f, weighted = 0.0f, term = 0.0f;
                each_of<kSteps + 3>([&](auto step) {
                    constexpr int n = decltype(step)::value, set = n / 16;
                    if constexpr (n % 16 == 0 && set + 1 < kSteps / 16) sets[(set + 1) & 1] = products((set + 1) / 4, (set + 1) % 4);
                    if constexpr (n >= 3) acc = acc + term;
                    if constexpr (n >= 2 && n < kSteps + 2) term = round_bf16(weighted);
                    if constexpr (n >= 1 && n < kSteps + 1) weighted = clamped * wv[(n - 1) / 4 % 16][(n - 1) % 4];
                    if constexpr (n < kSteps && n % 16 == 0) {
                        clamped = relu_bf16(sets[set & 1][0]);
                        asm volatile("" : "+v"(clamped), "+v"(sets[set & 1]));  // the other fifteen, now that this one was waited for
                    } else if constexpr (n < kSteps) {
                        clamped = clamp_bf16(sets[set & 1][n % 16]);
                    }
                    if constexpr (n == kPairHeads + 2 || n == kSteps + 2) asm volatile("" : "+v"(acc));
                    if constexpr (n == kPairHeads + 2) finish(0, info[0]);
                    if constexpr (n == kSteps + 2) finish(1, info[1]);
                    __builtin_amdgcn_sched_barrier(0);
                });
            } else {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    if (!take[u]) continue;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        if (c * 16 >= heads) break;
                        const f32x16 d = products(u, c);
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc = acc + head_term(d[i], wv[4 * c + i / 4][i % 4]);
                    }
                    finish(u, info[u]);
                }
            }
        }
        if (tile + 2 < tiles) park(buf ^ 1, 0), park(buf ^ 1, 1);
    }
    if (lane < 2) sh.left[wave][lane] = lane ? left[1] : left[0];
    __syncthreads();
    bool some_left = false;
#pragma unroll
    for (int i = 0; i < kPairWaves; ++i) some_left = some_left || (sh.left[i][0] | sh.left[i][1]) != 0;
    return some_left;
}

// Rows that are codes go through the fp4 instruction; of the others nothing that those needed is kept.
__global__ __launch_bounds__(kPairThreads, 2) void score_blocks_codes_kernel(const PairArgs args) {
    __shared__ PairShared<true> sh;
    int tid = threadIdx.x;
    {
        const PairPlace at = pair_place(args, tid);
        if (!at.tiles) return;  // workgroup-uniform
        if (!score_codes(args, at, sh)) return;
    }
    asm volatile("" : "+v"(tid));
    score_left<false>(args, pair_place(args, tid), sh);
}

// Few queries (a decode step: one). A workgroup owns one query's 64 heads against 32 HT blocks, a
// wave 16 HT heads and 32 blocks of them: 16 x 16 matrix tiles, operands straight from memory (lane
// group g holds the eight dims at 32 j + 8 g of row n16: four lanes take a line of a row, where a
// lane per row takes a line each), the head terms through LDS, the first wave folding them in head
// order. Bound by latency. 8 192 blocks: 14.1 us with every dot folded term by term, 8.0 as 32 x 32
// tiles of 64-block workgroups with a lane per row, 6.0 so.
constexpr int kOneThreads = 4 * kWave;
template <int HT>
__global__ __launch_bounds__(kOneThreads) void score_blocks_one_kernel(
    const float* __restrict__ q, const float* __restrict__ kv, const float* __restrict__ w,
    float* __restrict__ score, int s, int n_comp, int heads, int ratio) {
    constexpr int BLOCKS = 32 * HT;
    __shared__ float terms[kPairHeads][BLOCKS];
    __shared__ int inexact;
    const int lane = threadIdx.x & (kWave - 1), g = lane >> 4, n16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int t = blockIdx.y;
    const long long cw = (long long)blockIdx.x * BLOCKS, c = cw + (lane & (BLOCKS - 1));
    if (first_query(t, t + 1, ratio, cw & ~63ll) > t) return;  // workgroup-uniform: no block of the 64 is legal for t
    if (threadIdx.x == 0) inexact = 0;
    const size_t base = (size_t)t * heads;
    const int h0 = HT == 1 ? wave * 16 : (wave & 1) * 32, c0 = HT == 1 ? 0 : (wave >> 1) * 32;
    __syncthreads();
    if (h0 < heads) {
        struct Row {
            f32x4 v[8];
        };
        const auto fetch = [&](const float* p) {
            Row r;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                r.v[2 * j] = *reinterpret_cast<const f32x4_u*>(p + 32 * j + 8 * g);
                r.v[2 * j + 1] = *reinterpret_cast<const f32x4_u*>(p + 32 * j + 8 * g + 4);
            }
            return r;
        };
        const auto operand = [&](const Row& r, bool live, bf16x8 (&x)[4]) {
            RowSpan span;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                u32x4 b;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    f32x4 u = r.v[2 * k + j];
                    if (!live) u = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    b[2 * j] = upper_halves(u.x, u.y), b[2 * j + 1] = upper_halves(u.z, u.w);
                    span.add(b[2 * j], low_half_bits(u));
                    span.add(b[2 * j + 1], 0);
                }
                x[k] = __builtin_bit_cast(bf16x8, b);
            }
            uint32_t f = span.folded();
            f = span_max(f, __shfl_xor(f, 16, kWave));
            return span_of(span_max(f, __shfl_xor(f, 32, kWave)));
        };
        const long long last = n_comp - 1;
        Row rq[HT], rk[2];
        float wv[HT][4];
#pragma unroll
        for (int u = 0; u < HT; ++u) rq[u] = fetch(q + (base + min(h0 + 16 * u + n16, heads - 1)) * 128);
#pragma unroll
        for (int u = 0; u < 2; ++u) rk[u] = fetch(kv + (size_t)min(cw + c0 + 16 * u + n16, last) * 128);
#pragma unroll
        for (int u = 0; u < HT; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) wv[u][i] = w[base + min(h0 + 16 * u + 4 * g + i, heads - 1)];
        bf16x8 a[HT][4], b[2][4];
        int q_span = 0;
#pragma unroll
        for (int u = 0; u < HT; ++u) q_span = max(q_span, operand(rq[u], h0 + 16 * u + n16 < heads, a[u]));
        const int k_span = max(operand(rk[0], true, b[0]), operand(rk[1], true, b[1]));
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) q_span = max(q_span, __shfl_xor(q_span, m, kWave));
        if (__any(q_span + k_span > kExactSpan)) {
            if (lane == 0) inexact = 1;
        } else {
#pragma unroll
            for (int v = 0; v < 2 * HT; ++v) {
                f32x4 d = {0, 0, 0, 0};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[v >> 1][k], b[v & 1][k], d, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int hh = h0 + 16 * (v >> 1) + 4 * g + i;
                    if (hh < heads) terms[hh][c0 + 16 * (v & 1) + n16] = head_term(d[i], wv[v >> 1][i]);
                }
            }
        }
    }
    __syncthreads();
    if (inexact) {  // term by term: every wave a quarter of the heads
        const int per = (heads + 3) / 4, g0 = min(wave * per, heads), g1 = min(g0 + per, heads);
        float row_v[128];
        load_row(row_v, kv + (size_t)(c < n_comp ? c : n_comp - 1) * 128);
        if constexpr (HT == 1) {  // each half of the wave half of those (of an odd number the middle one twice)
            const int n = (g1 - g0 + 1) / 2, first = lane < 32 ? g0 : g1 - n;
            if (n > 0)
                fold_heads<false>(q + (base + first) * 128, w + base + first, n, row_v,
                                  [&](int i, float term) { terms[first + i][lane & (BLOCKS - 1)] = term; });
        } else {
            walk_pairs(q, w, row_v, base + g0, base + g1, [&](size_t h, float term) { terms[h - base][lane] = term; });
        }
        __syncthreads();
    }
    if (threadIdx.x < BLOCKS) {
        float acc = 0.0f;
        for (int hh = 0; hh < heads; ++hh) acc = acc + terms[hh][lane];
        if (c < n_comp) score[(size_t)t * n_comp + c] = round_bf16(acc);
    }
}

// Any other width: the block's row is re-read through the vector cache for every head.
__global__ __launch_bounds__(kScoreThreads) void index_score_blocks_any_kernel(
    const float* __restrict__ q, const float* __restrict__ kv, const float* __restrict__ w,
    float* __restrict__ score, int s, int n_comp, int heads, int hd, int t_per_group, int ratio) {
    const long long c = (long long)block_group(ratio) * kScoreThreads + threadIdx.x;
    const float* const kvr = kv + (size_t)(c < n_comp ? c : n_comp - 1) * hd;
    const int t1 = min(s, query_group(ratio) * t_per_group + t_per_group);
    const long long cw = (long long)block_group(ratio) * kScoreThreads +
                         (__builtin_amdgcn_readfirstlane((int)threadIdx.x) & ~(kWave - 1));
    const int t0 = first_query(query_group(ratio) * t_per_group, t1, ratio, cw);
    for (int t = t0; t < t1; ++t) {
        float acc = 0.0f;
        for (int hh = 0; hh < heads; ++hh) {
            const float* const qh = q + ((size_t)t * heads + hh) * hd;  // wave-uniform
            float dot = 0.0f;
            for (int i = 0; i < hd; ++i) {
                const float prod = qh[i] * kvr[i];
                dot = dot + prod;
            }
            acc = acc + head_term(dot, w[(size_t)t * heads + hh]);
        }
        if (c < n_comp) score[(size_t)t * n_comp + c] = round_bf16(acc);
    }
}

}  // namespace rk

extern "C" int rivoli_act_quant_f4_rotated(float* x, int rows, int d, void* stream) {
    if (rows <= 0 || d <= 0) return 1001;
    if (d > rk::kSpreadMaxD) return 1002;
    if (d & (d - 1)) return 1003;
    if (d % 32) return 1004;
    if (!x) return 1001;
    if (!rk::aligned16(x)) return 1004;  // rows are moved 16 bytes at a time
    (void)hipGetLastError();
    const float scale = 1.0f / std::sqrt((float)d);
    const int lpr = d / 4;
    const long long rows_per_step = (long long)(rk::kWave / lpr) * (rk::kSpreadThreads / rk::kWave);
    const bool few = rows <= rows_per_step * rk::kSpreadInFlight * rk::kSpreadFewGroups;
    const long long rows_per_group = few ? rows_per_step : rows_per_step * rk::kSpreadInFlight;
    const dim3 grid((unsigned)((rows + rows_per_group - 1) / rows_per_group)), block(rk::kSpreadThreads);
    hipStream_t st = (hipStream_t)stream;
#define RK_SPREAD(LPR)                                                                                      \
    if (few)                                                                                                \
        rk::launch_kernel((rk::f4_rotated_kernel<LPR, 1>), grid, block, 0, st, x, (long long)rows, scale);  \
    else                                                                                                    \
        rk::launch_kernel((rk::f4_rotated_kernel<LPR, rk::kSpreadInFlight>), grid, block, 0, st, x,         \
                          (long long)rows, scale)
    switch (lpr) {
        case 8: RK_SPREAD(8); break;
        case 16: RK_SPREAD(16); break;
        case 32: RK_SPREAD(32); break;
        default: RK_SPREAD(64); break;
    }
#undef RK_SPREAD
    return rk::launch_status();
}

namespace rk {
static int score_blocks_launch(const float* q, const float* kv, const float* w, float* score, int s,
                               int n_comp, int heads, int hd, int ratio, hipStream_t st) {
    if (s <= 0 || heads <= 0 || hd <= 0) return 1001;
    // refused, not an empty success: the reference produces no score tensor at all before the
    // first block completes (blockindex.hip:268-273)
    if (n_comp <= 0) return 1005;
    if (!q || !kv || !w || !score) return 1001;
    (void)hipGetLastError();
    if (hd == 128 && aligned16(kv) && heads <= kPairHeads) {
        const ScorePlan plan = score_plan(s, n_comp);
        const PairArgs args = {q, kv, w, score, s, n_comp, heads, plan.split, ratio};
        const dim3 grid(plan.groups, plan.rows);
        switch (plan.kernel) {
            case ScoreKernel::kOne32:
                rk::launch_kernel(score_blocks_one_kernel<1>, dim3((unsigned)(((long long)n_comp + 31) / 32), (unsigned)s),
                                  dim3(kOneThreads), 0, st, q, kv, w, score, s, n_comp, heads, ratio);
                return launch_status();
            case ScoreKernel::kOne64:
                rk::launch_kernel(score_blocks_one_kernel<2>, dim3((unsigned)(((long long)n_comp + 63) / 64), (unsigned)s),
                                  dim3(kOneThreads), 0, st, q, kv, w, score, s, n_comp, heads, ratio);
                return launch_status();
            case ScoreKernel::kCodes:
                rk::launch_kernel(score_blocks_codes_kernel, grid, dim3(kPairThreads), 0, st, args);
                return launch_status();
            case ScoreKernel::kPair:
                rk::launch_kernel(score_blocks_pair_kernel, grid, dim3(kPairThreads), 0, st, args);
                return launch_status();
            case ScoreKernel::kNone:
                break;
        }
    }
    // enough workgroups to fill the part while a workgroup keeps its rows for several queries
    const unsigned c_groups = (unsigned)(((long long)n_comp + kScoreThreads - 1) / kScoreThreads);
    int t_per_group = kScoreQueriesPerGroup;
    while (t_per_group > 1 && (long long)c_groups * ((s + t_per_group - 1) / t_per_group) < 2048) t_per_group >>= 1;
    if (ratio <= 0)
        while ((s + t_per_group - 1) / t_per_group > 65535) t_per_group <<= 1;  // the grid's second extent
    const unsigned t_groups = (unsigned)((s + t_per_group - 1) / t_per_group);
    if (ratio > 0 && c_groups > 65535u) return 1002;  // more than 2^24 blocks
    const dim3 grid = ratio > 0 ? dim3(t_groups, c_groups) : dim3(c_groups, t_groups);
    const dim3 block(kScoreThreads);
    if (hd == 128 && aligned16(kv) && (long long)s * c_groups < 256 && heads <= kSplitMaxHeads) {
        const unsigned groups = (unsigned)(((long long)n_comp + kWave - 1) / kWave);
        rk::launch_kernel(index_score_blocks_128_split_kernel, dim3(groups), dim3(kSplitWavesPerGroup * kWave),
                          (size_t)heads * kWave * sizeof(float), st, q, kv, w, score, s, n_comp, heads, ratio);
        return launch_status();
    }
    if (hd == 128 && aligned16(kv))
        rk::launch_kernel(index_score_blocks_128_kernel, grid, block, 0, st, q, kv, w, score, s, n_comp,
                          heads, t_per_group, ratio);
    else
        rk::launch_kernel(index_score_blocks_any_kernel, grid, block, 0, st, q, kv, w, score, s, n_comp,
                          heads, hd, t_per_group, ratio);
    return launch_status();
}
}  // namespace rk

extern "C" int rivoli_index_score_blocks(const float* q, const float* kv, const float* w,
                                         float* score, int s, int n_comp, int heads, int hd,
                                         void* stream) {
    return rk::score_blocks_launch(q, kv, w, score, s, n_comp, heads, hd, 0, (hipStream_t)stream);
}

extern "C" int rivoli_index_score_blocks_prefill(const float* q, const float* kv, const float* w,
                                                 float* score, int s, int n_comp, int heads, int hd,
                                                 int ratio, void* stream) {
    if (ratio <= 0) return 1001;
    return rk::score_blocks_launch(q, kv, w, score, s, n_comp, heads, hd, ratio, (hipStream_t)stream);
}
