// Attention over an index list at d = 512 for calls that fill the part (more than 256 workgroups
// of 64 heads): the kernel that gather_attn.hip launches for a prompt's queries.
//
// What bounds it: the matrix cores' time (96 instructions of 32 cycles a wave and tile of 32 slots)
// and, beside them, the instruction issue of a lone wave, 5 cycles an instruction. So a wave owns as
// much of a tile as its registers hold: 32 heads over all 512 dims and all 512 columns, one wave a
// SIMD, 128 registers of query, 256 of sums (the accumulation registers). Nothing is exchanged between
// waves (the kernel of 16 heads and half the dims a wave exchanges scores at a barrier every tile and
// runs every softmax twice), a row is read from LDS once for 32 heads instead of 16, and the two
// waves of a workgroup (64 heads) share only the staging of its rows. 66.5 KB of LDS: two workgroups a
// compute unit, one in its prologue or epilogue beside the other's tiles.
// 8192 queries x 640 slots of 64 heads: 1624 us -> 1045 us, of late 1064 -> 1040 with 32 of a tile's 290 vector instructions less (a
// conversion for two weights, row addresses from scalar registers). Its 0.94 P of products (the weights' remainders counted)
// run at 0.90 P/s; a large bf16 product sustains 1.40 here, at 1.97 GHz, where power limits it. This kernel is held to
// 2.15 GHz by the same limit (2.4 before), so what is left to save in cycles is worth half of it in time.
//
// A matrix instruction holds its unit for 32 cycles, in which the wave issues about six others: what a
// tile needs besides (operand reads, the next tile's rows, the second half of the weights) is
// cut into steps of two or three instructions and dealt out one behind each. As bursts of whole rows the same
// work took 1123 us, with the query's and the results' rows scattered 1464.
#pragma once
#include <type_traits>
#include <utility>

#include "attend_common.hpp"

namespace rk {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kGwThreads = 128;                 // two waves, 32 heads each
constexpr int kGwHeads = 32;
constexpr int kGwTile = 32;                     // slots a tile
constexpr int kGwRowsPerWave = kGwTile / 2;     // rows of a tile that a wave stages
constexpr int kGwKSteps = kGaD / 16;            // 32 steps of the score contraction
constexpr int kGwColTiles = kGaD / 32;          // 16 output column tiles
constexpr int kGwRing = 4;                      // rows on their way to a wave: 32 registers
constexpr int kGwSmemBytes = 2 * kGaTileBytes + 16;
static_assert(2 * kGwSmemBytes <= 160 * 1024, "two workgroups a compute unit");
// The reference maximum of a head is a tile's maximum (log2 units), moved when a later maximum passes it by kGwGrow:
// moving it scales 256 sums through ordinary registers (6000 cycles, more than a tile), and a window of 8, the
// other kernels', moves it for every outlier row. A head's largest weight lies in 2^0 .. 2^100, as hi + lo of its own exponent and so
// within 2^-18 of itself; it is seldom a power of two as the other kernels' is, so the denominator sums hi and lo too (results
// that are not the nearest bf16, 3000 queries with outlier rows: 6.3e-4 of them where it summed the weights, 5.5e-4 so and with the
// kernel of 64 heads; 0.5 % of the time). What the window costs is range: sums of weights of 2^100 overflow where
// |kv| passes 2^17. Such a query is done again with the window of 8, and gives what the other kernels give.
constexpr float kGwGrow = 100.0f;

// Row of a tile buffer (1040 bytes a row) that holds slot s: sixteen lanes of a 16-byte read (slots 0-3, 12-15, 20-23,
// 24-27, then the rest) meet in no bank, and so do the four slots of a transposing read, 64 bytes each.
__device__ __forceinline__ constexpr int gw_row_of_slot(int s) { return (s & 16) | 4 * (s & 3) | ((s >> 2) & 3); }

template <class F, int... I>
__device__ __forceinline__ void unrolled_steps(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unrolled(F&& f) {
    unrolled_steps(f, std::make_integer_sequence<int, N>{});
}

typedef const __attribute__((address_space(1))) char* global_bytes;

struct GwRow {  // a row on its way: dims 4 lane .. and 256 + 4 lane ..
    f32x4 v[2];
    __device__ __forceinline__ void ask(global_bytes row, int lane) { ask_at(row, 16u * lane); }
    __device__ __forceinline__ void ask_at(global_bytes row, uint32_t at) {
        v[0] = *(const __attribute__((address_space(1))) f32x4*)(row + at);
        v[1] = *(const __attribute__((address_space(1))) f32x4*)(row + at + 1024);
    }
    __device__ __forceinline__ u32x4 bf16() const {
        return u32x4{pack_bf16x2(v[0].x, v[0].y), pack_bf16x2(v[0].z, v[0].w),
                     pack_bf16x2(v[1].x, v[1].y), pack_bf16x2(v[1].z, v[1].w)};
    }
    __device__ __forceinline__ uint32_t bits() const {
        uint32_t any = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) any |= __float_as_uint(v[i >> 2][i & 3]);
        return any;
    }
};
struct GwEntries {  // a tile's row addresses, slot n32's in lanes n32 and n32 + 32
    uint32_t lo, hi;
};

// A list's tiles. The addresses of masked slots are those of a live row of the query: its weight there is 0
// and nothing that no slot lists is read (but row 0, in place of a list that is masked throughout).
struct GwList {
    const int* ix;
    uint64_t kv;
    int topk, n_kv;
    int end_tile, safe;
    __device__ __forceinline__ int fetch(int n32, int tile) const {
        return ix[min((unsigned)tile * kGwTile + n32, (unsigned)topk - 1)];
    }
    __device__ __forceinline__ GwEntries entries(int n32, int tile, int p, uint32_t& mask) const {
        const unsigned pos = (unsigned)tile * kGwTile + n32;
        const bool live = tile < end_tile && pos < (unsigned)topk && (unsigned)p < (unsigned)n_kv;
        mask = (uint32_t)__builtin_amdgcn_ballot_w64(live);
        const uint64_t at = kv + ((uint64_t)(unsigned)(live ? p : safe) << 11);
        return GwEntries{(uint32_t)at, (uint32_t)(at >> 32)};
    }
};

// A wave's 32 heads (qh, B operand fragments) over the whole list, results to o. False where the workgroup's
// results are not all in range and a narrower window may have them so.
template <int PSPLIT>
__device__ __forceinline__ bool gather_attn_wide_pass(const GatherAttnArgs& a, lds_ptr<uint8_t> kr, size_t t, int head0,
                                                      const bf16x8 (&qh)[kGwKSteps], const GwList& list,
                                                      int f0, int f1, int f2, float window) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // what the lane's number gives is worked out here, not kept through the prologue
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5, n32 = lane & 31, n16 = lane & 15;
    auto row_address = [&](const GwEntries& e, int i) -> global_bytes {  // the wave's row i of a tile
        const uint32_t lo = __builtin_amdgcn_readlane(e.lo, kGwRowsPerWave * wave + i);
        const uint32_t hi = __builtin_amdgcn_readlane(e.hi, kGwRowsPerWave * wave + i);
        return (global_bytes)(uintptr_t)((uint64_t)hi << 32 | lo);
    };
    auto deposit = [&](int buf, int slot, u32x4 v) {
        *(lds_ptr<u32x4>)(kr + buf * kGaTileBytes + gw_row_of_slot(slot) * kGaRowBytes + 16 * lane) = v;
    };

    uint32_t m_cur, m_next, m_after;  // live slots of this tile and the two after it
    const GwEntries e_first = list.entries(n32, 0, f0, m_cur);
    GwEntries e_next = list.entries(n32, 1, f1, m_next), e_after = list.entries(n32, 2, f2, m_after);
    // O^T: a lane holds four neighbouring columns of one head in each quarter of a tile, so what scales a head
    // is a register of its own lane. Kept in the accumulation registers ("a") throughout: 256 of them, all there are.
    f32x16 o[kGwColTiles];
    GwRow raw[kGwRing];
#pragma unroll
    for (int b = 0; b < kGwRowsPerWave; b += 8) {
        GwRow r[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i].ask(row_address(e_first, b + i), lane);
        __builtin_amdgcn_sched_barrier(0);
        if (b == 0) {  // while the first rows are on their way
            const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int c = 0; c < kGwColTiles; ++c)  // zeros at a sixteenth of the instructions of writing them
                asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %1, 0" : "=a"(o[c]) : "v"(z));
            // The compiler keeps no distance from assembly: a query without a live slot, which reads them first of all, does so far behind the
            // deposits below.
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) deposit(0, kGwRowsPerWave * wave + b + i, r[i].bf16());
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < kGwRing; ++i) raw[i].ask(row_address(e_next, i), lane);
    __syncthreads();

    float m_ref = -INFINITY, l_sum = 0.0f;
    const float qs = fabsf(a.qscale);  // its sign is in the query

    // A lane's place in a row, made anew at the head of each stretch without a branch: only within one does the compiler see 32 bits of
    // it and take a row's address from scalar registers (else a 64-bit addition a row).
    uint32_t lane_at = 16u * lane;
    for (int tile = 0; tile < list.end_tile; ++tile) {
        asm volatile("" : "+v"(lane_at));
        const int fetched = list.fetch(n32, tile + 3);
        const int buf = tile & 1;
        const lds_ptr<uint8_t> krb = kr + buf * kGaTileBytes;
        // The next tile's rows, four steps a row: its values (asked for kGwRing rows ago) to LDS as bf16, the row
        // kGwRing further on asked for in their registers. (The half asked for last first: one wait for both.)
        u32x4 staged = {0u, 0u, 0u, 0u};
        global_bytes row_at = nullptr;
        auto row_step = [&](auto kc) {
            constexpr int k = decltype(kc)::value, i = k / 4, part = k % 4;
            if constexpr (k >= 0 && k < kGwRowsPerWave * 4) {
                GwRow& r = raw[i % kGwRing];
                if constexpr (part == 0) staged.z = pack_bf16x2(r.v[1].x, r.v[1].y), staged.w = pack_bf16x2(r.v[1].z, r.v[1].w);
                if constexpr (part == 1) {
                    constexpr int next = i + kGwRing;
                    row_at = next < kGwRowsPerWave ? row_address(e_next, next) : row_address(e_after, next - kGwRowsPerWave);
                    staged.x = pack_bf16x2(r.v[0].x, r.v[0].y);
                }
                if constexpr (part == 2) {
                    staged.y = pack_bf16x2(r.v[0].z, r.v[0].w);
                    deposit(buf ^ 1, kGwRowsPerWave * wave + i, staged);
                }
                if constexpr (part == 3) r.ask_at(row_at, lane_at);
            }
        };

        // ---- scores: S^T[slot][column], the tile's rows as A. Written as assembly because the sums of the scores
        // have to be ordinary registers while o's are accumulation registers. What the compiler would see to is
        // seen to here: the operands come from LDS reads and from qh, no vector instruction writes one
        // within two instructions before its product (tests/test_kernel_resources.py reads the listing for that), and the
        // wait states between the last product and the first use of s are the s_nop below.
        f32x16 s;
        {
            const lds_ptr<bf16x8> ap = (lds_ptr<bf16x8>)(krb + gw_row_of_slot(n32) * kGaRowBytes + 16 * g);
            bf16x8 f[6];  // three pairs: one in the products, two on their way
#pragma unroll
            for (int i = 0; i < 4; ++i) f[i] = ap[2 * i];
            unrolled<kGwKSteps>([&](auto jc) {
                constexpr int j = decltype(jc)::value, k = j ^ 1;  // a pair's second first: one wait for both
                if constexpr (j == 0)
                    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(f[k % 6]), "v"(qh[k]));
                else
                    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(f[k % 6]), "v"(qh[k]));
                if constexpr (j + 4 < kGwKSteps) f[(j + 4) % 6] = ap[2 * (j + 4)];
                row_step(jc);
                __builtin_amdgcn_sched_barrier(0);
            });
            asm volatile("s_nop 15\n\ts_nop 2" : "+v"(s));
        }
        // ---- online softmax: the lane's 16 slots are 8 (i >> 2) + 4 g + (i & 3) of head n32
        if (m_cur != 0xffffffffu) {
            const uint32_t mine = m_cur >> (4 * g);
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = (mine >> (8 * (i >> 2) + (i & 3))) & 1 ? s[i] : -INFINITY;
        }
        float tmax = s[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) tmax = fmaxf(tmax, s[i]);
        {
            auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
            tmax = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1])) * qs;
        }
        const bool grow = tmax > m_ref + window;  // false while everything is masked
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
            const float corr = grow ? __builtin_amdgcn_exp2f(m_ref - tmax) : 1.0f;  // 2^-inf = 0 at first
            if (grow) m_ref = tmax;
            l_sum *= corr;
#pragma unroll
            for (int c = 0; c < kGwColTiles; ++c) {
                asm volatile("" : "+a"(o[c]));
                f32x16 x = o[c];
#pragma unroll
                for (int i = 0; i < 16; ++i) x[i] *= corr;
                asm volatile("" : "+a"(x));
                o[c] = x;
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const float mu = m_ref == -INFINITY ? 0.0f : m_ref;
        // p[ks][j] is slot 16 ks + 8 (j >> 2) + 4 g + (j & 3): the score registers in order are the value product's
        // B operand, so a weight never leaves its lane. The denominator sums what the products see, the rounded weights and their
        // remainders: a weight that is most of a head's comes out as 1 whatever its reference maximum.
        asm volatile("" : "+v"(lane_at));
        u32x4 p[2], p_lo[2];
        float e0 = 0.0f, e1 = 0.0f;
        auto weights = [&](auto ksc, auto pairc, auto partc) {  // two weights, in three steps
            constexpr int ks = decltype(ksc)::value, i = 2 * decltype(pairc)::value, part = decltype(partc)::value;
            if constexpr (part == 0) {
                e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * ks + i], qs, -mu));  // masked -> 0
                e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * ks + i + 1], qs, -mu));
            }
            if constexpr (part == 1) {
                uint32_t hi = pack_bf16x2(e0, e1);
                asm("" : "+v"(hi));  // (else a half that is taken out of the pair below is converted once more by itself)
                p[ks][i / 2] = hi;
            }
            if constexpr (part == 2) {
                const uint32_t hi = p[ks][i / 2];
                const uint32_t lo = PSPLIT == 2 ? pack_bf16x2(e0 - bf16_lo_to_f32(hi), e1 - bf16_hi_to_f32(hi)) : 0u;
                p_lo[ks][i / 2] = lo;
                typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
                l_sum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, hi), ones, l_sum, false);
                if (PSPLIT == 2) l_sum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, lo), ones, l_sum, false);
                asm volatile("" : "+v"(l_sum));  // summed here: sixteen weights kept for later are sixteen registers
            }
        };

        // ---- values: O^T[column][head] += V^T . P^T, the tile through the transposing read as A. A read hands a lane
        // four slots of one column; lane i of sixteen addresses slot i >> 2, columns 4 (i & 3) .. +3.
        const lds_ptr<uint8_t> vrow = krb + (4 * (n16 >> 2) + g) * kGaRowBytes + (16 * ((lane >> 4) & 1) + 4 * (n16 & 3)) * 2;
        auto value_frag = [&](int c, int ks) -> bf16x8 {
            typedef short s16x4 __attribute__((ext_vector_type(4)));
            typedef short s16x8 __attribute__((ext_vector_type(8)));
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<s16x4>)(vrow + 16 * ks * kGaRowBytes + 64 * c));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<s16x4>)(vrow + (16 * ks + 2) * kGaRowBytes + 64 * c));
            const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            return __builtin_bit_cast(bf16x8, both);
        };
        bf16x8 f[6];
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = value_frag(i, 0);
        __builtin_amdgcn_sched_barrier(0);
        unrolled<12>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            weights(std::integral_constant<int, 0>{}, std::integral_constant<int, i / 3>{}, std::integral_constant<int, i % 3>{});
        });
        // the weights of the second half of the slots, and the second half of the rows
        auto beside = [&](auto mc) {
            constexpr int m = decltype(mc)::value;
            if constexpr (m < 24 && m % 2 == 1)
                weights(std::integral_constant<int, 1>{}, std::integral_constant<int, m / 6>{}, std::integral_constant<int, (m % 6) / 2>{});
            else
                row_step(std::integral_constant<int, 32 + (m < 24 ? m / 2 : m - 12)>{});
        };
        unrolled<2 * kGwColTiles>([&](auto nc) {
            constexpr int n = decltype(nc)::value, x = n ^ 1, c = x % kGwColTiles, ks = x / kGwColTiles;
            o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[x % 6], __builtin_bit_cast(bf16x8, p[ks]), o[c], 0, 0, 0);
            beside(std::integral_constant<int, 2 * n>{});
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (PSPLIT == 2) o[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[x % 6], __builtin_bit_cast(bf16x8, p_lo[ks]), o[c], 0, 0, 0);
            if constexpr (n + 4 < 2 * kGwColTiles) f[(n + 4) % 6] = value_frag((n + 4) % kGwColTiles, (n + 4) / kGwColTiles);
            beside(std::integral_constant<int, 2 * n + 1>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        e_next = e_after, m_cur = m_next, m_next = m_after;
        e_after = list.entries(n32, tile + 3, fetched, m_after);
        __syncthreads();  // the next tile is staged, this one is read
    }

    // ---- the sink joins the denominator, the quotient is rounded to bf16
    {
        auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_sum), __float_as_uint(l_sum), false, false);
        l_sum = __uint_as_float(both[0]) + __uint_as_float(both[1]);
    }
    const int head = head0 + n32;
    const float sk = a.sink[head < a.h ? head : 0] * kLog2e;
    // in units of 2^max(m_ref, sk); nothing live: m_ref is still -inf and the output NaN
    const float fit = sk > m_ref ? exp2f(m_ref - sk) : 1.0f;
    const float l = m_ref == -INFINITY ? NAN : l_sum * fit + (sk > m_ref ? 1.0f : exp2f(sk - m_ref));
    const float l_inv = fit / l;  // one division a head: the product's error is far below the bf16 rounding that follows
    // Out through the wave's own buffer, a head's 1 KiB a row, so that whole lines are stored (a lane's own four
    // columns at a time measured 2 us more a workgroup). Columns 32 c + 8 u + 4 g .. +3 of the products are dims
    // 4 (4 c + u) + 256 g .. +3: a staged row holds dims 4 lane .. and 256 + 4 lane .. side by side.
    const lds_ptr<uint8_t> own = kr + wave * kGaTileBytes;
    float most = 0.0f;  // the largest result, NaN where one is (the instruction takes three operands: half of one a result)
#pragma unroll
    for (int c = 0; c < kGwColTiles; ++c) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = o[c][4 * u + i] * l_inv;
#pragma unroll
            for (int i = 0; i < 4; i += 2)
                most = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(x[i]), fabsf(x[i + 1])), most);
            const u32x2 w = {pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
            *(lds_ptr<u32x2>)(own + n32 * kGaRowBytes + 8 * (4 * c + u) + 512 * g) = w;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    float* const out = a.o + t * a.h * kGaD;
#pragma unroll 8
    for (int r = 0; r < kGwHeads; ++r) {
        if (head0 + r >= a.h) break;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const u32x2 w = *(lds_ptr<u32x2>)(own + r * kGaRowBytes + 512 * k + 8 * lane);
            reinterpret_cast<f32x4*>(out + (size_t)(head0 + r) * kGaD)[64 * k + lane] =
                f32x4{bf16_lo_to_f32(w.x), bf16_hi_to_f32(w.x), bf16_lo_to_f32(w.y), bf16_hi_to_f32(w.y)};
        }
    }
    // Sums that overflowed, or a sink so far above the reference maximum that the quotient's factor is no normal number.
    if (window == kLazyRescale || list.end_tile == 0) return true;
    const lds_ptr<int> over = (lds_ptr<int>)(kr + 2 * kGaTileBytes) + 2;
    const bool bad = __builtin_amdgcn_ballot_w64(!(most < INFINITY && l_inv >= 0x1p-126f)) != 0;
    if (lane == 0) over[wave] = bad;
    __syncthreads();  // (and both buffers are read)
    return __builtin_amdgcn_readfirstlane(over[0] | over[1]) == 0;
}

// QSPLIT 2 keeps what bf16 leaves of a query that is not bf16-valued. The model's query is (its rotary stores bf16,
// crates/backend/kernels/mla.hip:432), and only such a query's 64 heads fit the registers: others are marked, for
// gather_attn_marked_kernel (gather_attn.hip) to do. The mark is the block's first output element: results are bf16
// values, so no result has its bits. A head's row is looked at ahead of most of the rest, so that a call whose queries are of
// the other kind spends a round trip a workgroup here and a quarter of its rows' traffic (with half of them on their way by then
// 8192 such queries of 640 slots took 1777 us, so 1740; bf16-valued ones the same within 0.6 %). Two passes over the list
// in this kernel, 16 heads and their remainders a wave, took 1.24 to 1.5 times the kernel of half the dims.
constexpr uint32_t kGwMark = 0x7fc0a55au;
constexpr int kGwFirstRows = 8;  // of a wave's, asked for with the first look

template <int QSPLIT, int PSPLIT>
__device__ __forceinline__ bool gather_attn_wide_query(const GatherAttnArgs& a, lds_ptr<uint8_t> kr, float window) {
    const lds_ptr<int> flag = (lds_ptr<int>)(kr + 2 * kGaTileBytes);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // nothing of it is kept for a second time
    const size_t t = blockIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5, n32 = lane & 31;
    const int head0 = blockIdx.y * 64 + kGwHeads * wave;
    const global_bytes q_at = (global_bytes)(uintptr_t)(a.q + t * a.h * kGaD);
    uint32_t* const mark = reinterpret_cast<uint32_t*>(a.o + (t * a.h + blockIdx.y * 64) * kGaD);

    GwRow first;
    if (QSPLIT == 2) first.ask(q_at + (size_t)blockIdx.y * 64 * (kGaD * 4), lane);
    // Trailing masked slots make no tiles: a wave looks at the list's last 512 entries (and at the 512 before
    // them while all are masked). They and the first tiles' entries are on their way while the query is.
    GwList list{a.idxs + t * a.topk, (uint64_t)(uintptr_t)a.kv, a.topk, a.n_kv, 0, 0};
    int tail[8];
    auto tail_fetch = [&](int end) {
#pragma unroll
        for (int i = 0; i < 8; ++i) tail[i] = list.ix[max(end - 64 * (8 - i) + lane, 0)];
    };
    tail_fetch(a.topk);
    const int f0 = list.fetch(n32, 0), f1 = list.fetch(n32, 1), f2 = list.fetch(n32, 2);

    // a wave's 32 heads go through its buffer like a tile's rows
    uint32_t any = 0;
    auto ask_query = [&](auto& v, int r0) {
#pragma unroll
        for (int i = 0; i < (int)(sizeof(v) / sizeof(GwRow)); ++i) {  // a head past h reads head 0: its column goes nowhere
            const int hd = head0 + r0 + i < a.h ? head0 + r0 + i : 0;
            v[i].ask(q_at + (size_t)hd * (kGaD * 4), lane);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto stage_query = [&](const auto& v, int r0) {
#pragma unroll
        for (int i = 0; i < (int)(sizeof(v) / sizeof(GwRow)); ++i) {
            *(lds_ptr<u32x4>)(kr + wave * kGaTileBytes + gw_row_of_slot(r0 + i) * kGaRowBytes + 16 * lane) = v[i].bf16();
            any |= v[i].bits();
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    {
        GwRow few[kGwFirstRows];
        ask_query(few, 0);
        if (QSPLIT == 2 && __builtin_amdgcn_ballot_w64((first.bits() & 0xffffu) != 0) != 0) {  // the same in both waves
            if (threadIdx.x == 0) *mark = kGwMark;
            return true;
        }
        stage_query(few, 0);
    }
    {
        GwRow rest[kGwHeads - kGwFirstRows];
        ask_query(rest, kGwFirstRows);
        stage_query(rest, kGwFirstRows);
    }
    if (QSPLIT == 2) {
        const bool has = __builtin_amdgcn_ballot_w64((any & 0xffffu) != 0) != 0;
        if (lane == 0) flag[wave] = has;
    }
    bf16x8 qh[kGwKSteps];
    {
        const lds_ptr<u32x4> ap = (lds_ptr<u32x4>)(kr + wave * kGaTileBytes + gw_row_of_slot(n32) * kGaRowBytes + 16 * g);
        const uint32_t sign = a.qscale < 0.0f ? 0x80008000u : 0u;
#pragma unroll
        for (int j = 0; j < kGwKSteps; ++j) qh[j] = __builtin_bit_cast(bf16x8, ap[2 * j] ^ sign);
#pragma unroll
        for (int j = 0; j < kGwKSteps; ++j) asm volatile("" : "+v"(qh[j]));
    }

    int used = 0;
    for (int end = a.topk;;) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int pos = end - 64 * (8 - i) + lane;
            const uint64_t m = __builtin_amdgcn_ballot_w64(pos >= 0 && (unsigned)tail[i] < (unsigned)a.n_kv);
            if (m != 0) {
                const int top = 63 - __builtin_clzll(m);
                used = end - 64 * (8 - i) + top + 1;
                list.safe = __builtin_amdgcn_readlane(tail[i], top);
            }
        }
        end -= 512;
        if (used != 0 || end <= 0) break;
        tail_fetch(end);
    }
    list.end_tile = (used + kGwTile - 1) / kGwTile;
    __syncthreads();  // the query is read: the first tile may take its place
    if (QSPLIT == 2 && __builtin_amdgcn_readfirstlane(flag[0] | flag[1]) != 0) {
        if (threadIdx.x == 0) *mark = kGwMark;
        return true;
    }
    return gather_attn_wide_pass<PSPLIT>(a, kr, t, head0, qh, list, f0, f1, f2, window);
}

template <int QSPLIT, int PSPLIT>
__global__ __launch_bounds__(kGwThreads, 1) void gather_attn_wide_kernel(const GatherAttnArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[kGwSmemBytes];
    // (the second time from the query on: kept for it through the epilogue, its 128 registers would spill)
    for (float window = kGwGrow; !gather_attn_wide_query<QSPLIT, PSPLIT>(a, (lds_ptr<uint8_t>)smem, window);) window = kLazyRescale;
}

}  // namespace rk
