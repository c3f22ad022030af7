// The k best of one row of up to 16 384 scores, emitted in index order, by one workgroup of sixteen waves with
// a row's keys in registers (a wave owns a contiguous run, 64 keys a step).
//
// What bounds it: the steps that follow one another (few rows leave each a compute unit to itself): a round trip to
// memory, then LDS and barriers. There are four barriers. The keys' smallest and largest place a histogram of
// 2048 equal bins over the range that the keys really take (a row's scores share a few exponents: bins
// of leading bits had half of the keys' LDS atomics meet in a dozen addresses); every wave finds the pivot bin for
// itself from sixteen totals and the 128 bins that hold it; the bin's members, up to 64, are listed with their
// indices, and again every wave finds the threshold among them, and what the waves before it emit, for itself. A bin
// that holds more becomes the range of the next histogram (three more barriers), and one that cannot be
// divided holds equal keys, of which the first are taken.
// One query of 8192 scores (sums of a ReLU), 2048 selected: 11.0 us by a 10-bit histogram under the highest bit that differs,
// ordered candidates in LDS and three more histograms of 8 bits; 7.7 here. 8 queries of 16 384 12.9 -> 8.8, all scores equal 13.1 -> 5.7,
// bf16-valued 14.2 -> 12.7.
#pragma once
#include "topk_common.hpp"

namespace rk {

constexpr int kSfWaves = 16;
constexpr int kSfThreads = kSfWaves * kWave;
constexpr int kSfBits = 11;
constexpr int kSfBins = 1 << kSfBits;
constexpr int kSfCopies = 4;   // of a bin, by lane: equal scores in neighbouring lanes meet a quarter as often
constexpr int kSfList = kWave; // members of the pivot bin that are listed: up to one a lane
constexpr int kSfHistWords = (kSfBins + 1) * kSfCopies;  // one bin more for what is no element
constexpr int kSfFillAt = kSfHistWords + 2 * kSfList + 5 * kSfWaves;  // how far the list is filled
constexpr int kSfLdsWords = kSfFillAt + 4;
static_assert(kSfBins == 2 * kSfThreads && kSfCopies == 4, "a thread owns two bins of four words");

// min / max over the wave, as scalars
template <class OP>
__device__ __forceinline__ uint32_t wave_fold(uint32_t v, OP op) {
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x112, 0xf, 0xf, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x114, 0xf, 0xf, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x118, 0xf, 0xf, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xf, 0xf, false));  // row_bcast:15
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xf, 0xf, false));  // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, kWave - 1);
}

// The rest of select_few, with the row's keys in registers: key 0 where there is no element. GUARD: key 0 is also a
// live one's (no number's, of all NaNs one), so elements are told apart by their place; otherwise by 0 < base.
template <int ITEMS, bool GUARD>
__device__ __forceinline__ void select_few_keys(const uint32_t (&key)[ITEMS], int nt, int steps, int seg0, int limit, uint32_t base,
                                                uint32_t span, uint32_t kq, uint32_t* __restrict__ out, uint32_t* lds, uint32_t add) {
    uint32_t* const hist = lds;
    uint32_t* const l_key = lds + kSfHistWords;
    uint32_t* const l_idx = l_key + kSfList;
    uint32_t* const s_a = l_idx + kSfList;   // [16] the waves' minima
    uint32_t* const s_b = s_a + kSfWaves;    // [16] maxima
    uint32_t* const s_tot = s_b + kSfWaves;  // [16] counts of the bins that a wave owns
    // [16] their keys above the pivot bin, and in it. Words of their own: with one value in the row no barrier stands between
    // the waves' reading of the minima and maxima and these.
    uint32_t* const s_gt = s_tot + kSfWaves;
    uint32_t* const s_eq = s_gt + kSfWaves;
    uint32_t* const s_fill = lds + kSfFillAt;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // steps in fours: a branch a key costs more than the three keys too many
    constexpr int kGroup = ITEMS < 4 ? ITEMS : 4;
    auto each = [&](auto&& body) {
#pragma unroll
        for (int j0 = 0; j0 < ITEMS; j0 += kGroup) {
            if (j0 >= steps) break;
#pragma unroll
            for (int j = j0; j < j0 + kGroup; ++j) body(j);
        }
    };
    auto clear = [&] {
        reinterpret_cast<uint4*>(hist)[tid] = uint4{0u, 0u, 0u, 0u};
        reinterpret_cast<uint4*>(hist)[kSfThreads + tid] = uint4{0u, 0u, 0u, 0u};
    };
    auto count_of = [&](int bin) -> uint32_t {
        const uint4 c = reinterpret_cast<const uint4*>(hist)[bin];
        return c.x + c.y + c.z + c.w;
    };
    uint32_t need = kq;                                    // still to be taken from the keys base .. base + span
    uint32_t lo = base, hi = base, in_bin = (uint32_t)nt;  // the pivot bin's keys
    auto in_range = [&](int j) {
        if (GUARD) asm volatile("" : "+v"(limit));  // (tested anew: sixteen masks kept are 32 scalar registers)
        return key[j] - lo <= hi - lo && (!GUARD || j * kWave < limit);
    };
    uint32_t* const mine = hist + (lane & (kSfCopies - 1));
    bool first = true;
    while (span != 0) {
        const int shift = span >> kSfBits ? 32 - kSfBits - __builtin_clz(span) : 0;
        if (first && !GUARD) {
            // no branch a key: what is no element lies past the range (0 - base > span) and goes to a bin of its own
            each([&](int j) {
                const uint32_t at = key[j] - base;
                atomicAdd(&mine[(at <= span ? at >> shift : (uint32_t)kSfBins) * kSfCopies], 1u);
            });
        } else {
            hi = lo + span;
            each([&](int j) {
                if (in_range(j)) atomicAdd(&mine[((key[j] - base) >> shift) * kSfCopies], 1u);
            });
        }
        first = false;
        __syncthreads();
        {
            const uint32_t total = wave_total(wave_inclusive_sum(count_of(2 * tid) + count_of(2 * tid + 1)));
            if (lane == 0) s_tot[wave] = total;
        }
        __syncthreads();
        // counted from the highest bin down: the wave whose bins hold the need-th key, then the lane, then the bin
        const uint32_t t = lane < kSfWaves ? s_tot[kSfWaves - 1 - lane] : 0u;
        const uint32_t t_incl = wave_inclusive_sum(t);
        const int wl = __builtin_ctzll(__builtin_amdgcn_ballot_w64(t_incl >= need));
        uint32_t above = (uint32_t)__builtin_amdgcn_readlane((int)(t_incl - t), wl);
        const int top = 2 * ((kSfWaves - 1 - wl) * kWave + kWave - 1 - lane) + 1;
        const uint32_t m1 = count_of(top), m0 = count_of(top - 1);
        const uint32_t m_incl = wave_inclusive_sum(m1 + m0) + above;
        const int ml = __builtin_ctzll(__builtin_amdgcn_ballot_w64(m_incl >= need));
        above = (uint32_t)__builtin_amdgcn_readlane((int)(m_incl - m1 - m0), ml);
        uint32_t bin = (uint32_t)__builtin_amdgcn_readlane(top, ml);
        in_bin = (uint32_t)__builtin_amdgcn_readlane((int)m1, ml);
        if (above + in_bin < need) above += in_bin, in_bin = (uint32_t)__builtin_amdgcn_readlane((int)m0, ml), --bin;
        need -= above;                // 1 <= need <= in_bin
        lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(base + (bin << shift)));
        hi = lo + min((1u << shift) - 1u, base + span - lo);
        if (need == in_bin || in_bin <= (uint32_t)kSfList) break;
        // the bin's keys are the next range, from its smallest to its largest: 0 when they are all equal
        uint32_t a = ~0u, b = 0u;
        each([&](int j) {
            const bool in = in_range(j);
            a = min(a, in ? key[j] : ~0u);
            b = max(b, in ? key[j] : 0u);
        });
        a = wave_fold(a, [](uint32_t x, uint32_t y) { return min(x, y); });
        b = wave_fold(b, [](uint32_t x, uint32_t y) { return max(x, y); });
        if (lane == 0) s_a[wave] = a, s_b[wave] = b;
        __syncthreads();              // (and every wave has looked at the histogram)
        clear();
        lo = base = wave_fold(s_a[lane & (kSfWaves - 1)], [](uint32_t x, uint32_t y) { return min(x, y); });
        hi = wave_fold(s_b[lane & (kSfWaves - 1)], [](uint32_t x, uint32_t y) { return max(x, y); });
        span = hi - lo;
        __syncthreads();
    }
    // A bin that is taken whole has no members to choose from (and is not the lowest: a key is left over); neither
    // has one of equal keys, of which the first `need` are taken.
    const bool whole = need == in_bin;
    const bool listed = !whole && lo != hi;
    if (whole) hi = lo - 1u;
    {
        uint32_t gt = 0, eq = 0;
        each([&](int j) {
            gt += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(key[j] > hi));
            eq += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(in_range(j)));  // (no use when the bin is taken whole)
        });
        if (lane == 0) s_gt[wave] = gt, s_eq[wave] = eq;
        if (listed && eq != 0) {  // a place in the list for the wave's members: their order there is no matter
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(s_fill, eq);
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
            asm volatile("" : "+s"(lo));  // the tests again: kept from above, their masks are more than the scalar registers hold
            each([&](int j) {
                const bool in = in_range(j);
                const unsigned long long mask = __builtin_amdgcn_ballot_w64(in);
                if (in) l_key[at + lanes_below(mask)] = key[j], l_idx[at + lanes_below(mask)] = (uint32_t)(seg0 + j * kWave + lane);
                at += (uint32_t)__popcll(mask);
            });
        }
    }
    __syncthreads();
    // T: select key > T and the first `ties` (in index order) of key == T; run_gt, run_eq: how many of those the waves before hold
    uint32_t T = hi, ties = whole ? 0u : need;
    auto before = [&](const uint32_t* v) -> uint32_t {
        const uint32_t x = lane < wave ? v[lane & (kSfWaves - 1)] : 0u;
        return wave_total(wave_inclusive_sum(x));
    };
    uint32_t run_gt = before(s_gt), run_eq = 0, here_eq = 0;  // here_eq: this wave's keys == T, where there are ties
    if (listed) {
        const bool is = lane < (int)in_bin;
        const uint32_t k = is ? l_key[lane] - lo : 0u, i = is ? l_idx[lane] : ~0u;  // (past every wave's run)
        auto count = [&](bool of) { return (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(is && of)); };
        uint32_t p = 0;
        bool exact = false;
        // bits that no member has need no step: of scores rounded to bf16, the low sixteen
        uint32_t open = wave_fold(k, [](uint32_t x, uint32_t y) { return x | y; });
        while (open != 0 && !exact) {
            const uint32_t bit = 0x80000000u >> __builtin_clz(open);
            open ^= bit;
            const uint32_t cand = p | bit;
            const uint32_t c = count(k >= cand);
            if (c >= need) p = cand;
            exact = c == need;
        }
        if (exact) {  // the members from lo + p on are as many as needed
            T = lo + p - 1u, ties = 0;
        } else {      // lo + p is the need-th largest
            T = lo + p;
            ties = need - count(k > p);
            run_eq = count(k == p && i < (uint32_t)seg0);
            here_eq = count(k == p && i - (uint32_t)seg0 < (uint32_t)(steps * kWave));
        }
        run_gt += count((exact ? k >= p : k > p) && i < (uint32_t)seg0);
    } else if (!whole) {
        run_eq = before(s_eq);
        here_eq = s_eq[wave];
    }
    T = (uint32_t)__builtin_amdgcn_readfirstlane((int)T);
    ties = (uint32_t)__builtin_amdgcn_readfirstlane((int)ties);
    // What is no element has key 0, never above T. It can equal T only where T is 0, the lowest key: then all that lies before a tie
    // that is taken is taken too. In steps past a wave's run (they go in fours) such a one stands where the next wave's elements
    // do, and what it stores is the index that stands at that place of the output anyway; past the row's end nothing is left to take:
    // slot < kq drops it. The compare also keeps a wrong threshold from ever turning into a write outside the caller's buffer.
    if (ties == 0 || __builtin_amdgcn_readfirstlane((int)here_eq) == 0) {
        run_gt += min(run_eq, ties);
        each([&](int j) {
            const bool g = key[j] > T;
            const unsigned long long mg = __builtin_amdgcn_ballot_w64(g);
            const uint32_t slot = run_gt + lanes_below(mg);
            if (g && slot < kq) out[slot] = (uint32_t)(seg0 + j * kWave + lane) + add;
            run_gt += (uint32_t)__popcll(mg);
        });
        return;
    }
    each([&](int j) {
        const bool g = key[j] > T, e = key[j] == T;
        const unsigned long long mg = __builtin_amdgcn_ballot_w64(g), me = __builtin_amdgcn_ballot_w64(e);
        const uint32_t E = run_eq + lanes_below(me);
        const uint32_t slot = run_gt + lanes_below(mg) + min(E, ties);
        if ((g || (e && E < ties)) && slot < kq) out[slot] = (uint32_t)(seg0 + j * kWave + lane) + add;
        run_gt += (uint32_t)__popcll(mg);
        run_eq += (uint32_t)__popcll(me);
    });
}

// requires 1 <= kq < nt <= 1024 * ITEMS; lds (16-byte aligned) holds kSfLdsWords words. Writes out[0 .. kq).
template <int ITEMS, class KEY>
__device__ __forceinline__ void select_few(const float* __restrict__ s, int nt, uint32_t kq, uint32_t* __restrict__ out,
                                           uint32_t* lds, uint32_t add) {
    uint32_t* const s_a = lds + kSfHistWords + 2 * kSfList;
    uint32_t* const s_b = s_a + kSfWaves;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per_wave = ((nt + kSfThreads - 1) / kSfThreads) * kWave;
    const int steps = per_wave / kWave;
    const int seg0 = wave * per_wave;
    const int rem = nt - seg0;
    const int here = rem < per_wave ? rem : per_wave;  // may be none
    const int limit = here - lane;                     // element j exists iff j * 64 < limit

    // every load in flight before the first is used: an element past the row's end reads the row's last score
    uint32_t key[ITEMS];
    {
        constexpr int kGroup = ITEMS < 4 ? ITEMS : 4;
        float v[ITEMS];
        const float* const run = s + (here > 0 ? seg0 : 0);
#pragma unroll
        for (int j0 = 0; j0 < ITEMS; j0 += kGroup) {
            if ((j0 + kGroup) * kWave <= here) {
#pragma unroll
                for (int j = j0; j < j0 + kGroup; ++j) v[j] = run[j * kWave + lane];
            } else {
#pragma unroll
                for (int j = j0; j < j0 + kGroup; ++j) v[j] = s[min((uint32_t)(seg0 + lane + j * kWave), (uint32_t)(nt - 1))];
            }
        }
        reinterpret_cast<uint4*>(lds)[tid] = uint4{0u, 0u, 0u, 0u};
        reinterpret_cast<uint4*>(lds)[kSfThreads + tid] = uint4{0u, 0u, 0u, 0u};
        if (tid == 0) lds[kSfFillAt] = 0u;
        uint32_t lo = ~0u, hi = 0u;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const bool live = j * kWave < limit;
            key[j] = live ? KEY::of(v[j]) : 0u;
            lo = min(lo, live ? key[j] : ~0u);
            hi = max(hi, key[j]);
        }
        lo = wave_fold(lo, [](uint32_t a, uint32_t b) { return min(a, b); });
        hi = wave_fold(hi, [](uint32_t a, uint32_t b) { return max(a, b); });
        if (lane == 0) s_a[wave] = lo, s_b[wave] = hi;
    }
    __syncthreads();
    const uint32_t base = wave_fold(s_a[lane & (kSfWaves - 1)], [](uint32_t a, uint32_t b) { return min(a, b); });
    const uint32_t span = wave_fold(s_b[lane & (kSfWaves - 1)], [](uint32_t a, uint32_t b) { return max(a, b); }) - base;
    if (base != 0)
        select_few_keys<ITEMS, false>(key, nt, steps, seg0, limit, base, span, kq, out, lds, add);
    else
        select_few_keys<ITEMS, true>(key, nt, steps, seg0, limit, base, span, kq, out, lds, add);
}

}  // namespace rk
