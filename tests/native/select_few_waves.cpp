// The selection of one row (rivoli_amd/csrc/select_few.hpp) on the CPU: every lane of its sixteen waves a fiber, the lanes of
// a wave in step at each operation across them, and the waves in an order of the caller's between two barriers. On a GPU that
// order is nobody's to choose, so a result that depends on it is a race; here it is one on every run.
// The Makefile makes select_few_host.hpp of the kernel's own headers, without their includes and register hints.
#include <stdint.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <memory>
#include <numeric>
#include <random>
#include <vector>

namespace {

constexpr int kLanes = 64, kAllWaves = 16;
constexpr size_t kStack = 32 * 1024;

struct Lane {
    ucontext_t context;
    enum { kRuns, kAtWave, kAtBarrier, kDone } state = kRuns;
};
struct Wave {
    uint64_t given[2][kLanes];  // what the lanes brought to this operation and to the one before
    int arrived = 0, parity[kLanes] = {};
};
Lane lanes[kAllWaves * kLanes];
Wave waves[kAllWaves];
ucontext_t scheduler;
int current;                                   // the running fiber
struct { int x; } threadIdx;

void yield_as(decltype(Lane::state) s) {
    Lane& l = lanes[current];
    l.state = s;
    swapcontext(&l.context, &scheduler);
}
// Brings `v` to the wave's next operation; afterwards all lanes' values are there.
const uint64_t* together(uint64_t v) {
    Wave& w = waves[current / kLanes];
    const int lane = current % kLanes, p = w.parity[lane] ^= 1;
    w.given[p][lane] = v;
    if (++w.arrived < kLanes) {
        yield_as(Lane::kAtWave);
    } else {
        w.arrived = 0;
        for (int i = 0; i < kLanes; ++i)
            if (i != lane) lanes[current - lane + i].state = Lane::kRuns;
    }
    return w.given[p];
}

struct uint4 { uint32_t x, y, z, w; };
constexpr int kWave = kLanes;

int lane_id() { return current % kLanes; }
void __syncthreads() { yield_as(Lane::kAtBarrier); }
uint32_t atomicAdd(uint32_t* p, uint32_t v) { const uint32_t old = *p; *p += v; return old; }
uint32_t __float_as_uint(float x) { uint32_t u; memcpy(&u, &x, 4); return u; }
int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
template <class T> T min(T a, T b) { return a < b ? a : b; }
template <class T> T max(T a, T b) { return a > b ? a : b; }

unsigned long long __builtin_amdgcn_ballot_w64(bool b) {
    const uint64_t* g = together(b);
    unsigned long long m = 0;
    for (int i = 0; i < kLanes; ++i) m |= (unsigned long long)(g[i] & 1) << i;
    return m;
}
int __builtin_amdgcn_readlane(int v, int lane) { return (int)together((uint32_t)v)[lane]; }
int __builtin_amdgcn_readfirstlane(int v) { return (int)together((uint32_t)v)[0]; }
uint32_t __builtin_amdgcn_mbcnt_lo(uint32_t mask, uint32_t add) {
    const int l = lane_id();
    return add + (uint32_t)__builtin_popcount(l < 32 ? mask & ((1u << l) - 1u) : mask);
}
uint32_t __builtin_amdgcn_mbcnt_hi(uint32_t mask, uint32_t add) {
    const int l = lane_id();
    return add + (l < 32 ? 0u : (uint32_t)__builtin_popcount(mask & ((1u << (l - 32)) - 1u)));
}
int __builtin_amdgcn_update_dpp(int old, int v, int control, int, int, bool) {  // all rows and banks enabled
    const uint64_t* g = together((uint32_t)v);
    const int l = lane_id();
    int from = -1;
    if (control > 0x110 && control < 0x120) from = (l & 15) >= (control & 15) ? l - (control & 15) : -1;  // row_shr
    if (control == 0x142 && l >= 16) from = (l & ~15) - 1;                                                // row_bcast:15
    if (control == 0x143 && l >= 32) from = 31;                                                           // row_bcast:31
    return from < 0 ? old : (int)g[from];
}
uint32_t wave_inclusive_sum(uint32_t v) {
    const uint64_t* g = together(v);
    return std::accumulate(g, g + lane_id() + 1, 0u, [](uint32_t a, uint64_t b) { return a + (uint32_t)b; });
}
uint32_t wave_total(uint32_t inclusive) { return (uint32_t)__builtin_amdgcn_readlane((int)inclusive, kLanes - 1); }

#define __device__
#define __host__
#define __forceinline__ inline
#define __restrict__
#include "build/select_few_host.hpp"

struct Call {
    const float* scores;
    int nt, k, items, total_order;
    uint32_t *out, *lds, add;
} call;

template <int ITEMS>
void select() {
    if (call.total_order)
        rk::select_few<ITEMS, rk::TotalOrderKey>(call.scores, call.nt, (uint32_t)call.k, call.out, call.lds, call.add);
    else
        rk::select_few<ITEMS, rk::FoldedZeroKey>(call.scores, call.nt, (uint32_t)call.k, call.out, call.lds, call.add);
}
void lane_main() {
    threadIdx.x = current;
    switch (call.items) {
        case 1: select<1>(); break;
        case 2: select<2>(); break;
        case 8: select<8>(); break;
        default: select<16>(); break;
    }
    yield_as(Lane::kDone);
}

}  // namespace

// Runs the selection with the waves taken, between two barriers, in ascending order (order 0), descending (1) or one that
// is drawn anew at each barrier (other values seed it). Returns the barriers passed, or -1 where they never end.
extern "C" int select_few_waves(const float* scores, int nt, int k, int items, int total_order, uint32_t add, int order, uint32_t* out) {
    std::vector<uint32_t> lds(rk::kSfLdsWords + 4, 0xDEADBEEFu);
    call = {scores, nt, k, items, total_order, out, lds.data() + (4 - (uintptr_t)lds.data() / 4 % 4) % 4, add};
    std::unique_ptr<char[]> stacks(new char[sizeof(lanes) / sizeof(lanes[0]) * kStack]);
    for (int i = 0; i < kAllWaves * kLanes; ++i) {
        getcontext(&lanes[i].context);
        lanes[i].context.uc_stack.ss_sp = stacks.get() + i * kStack;
        lanes[i].context.uc_stack.ss_size = kStack;
        lanes[i].context.uc_link = nullptr;
        makecontext(&lanes[i].context, lane_main, 0);
        lanes[i].state = Lane::kRuns;
    }
    for (Wave& w : waves) w = Wave();
    std::mt19937 rng((unsigned)order);
    std::vector<int> turn(kAllWaves);
    std::iota(turn.begin(), turn.end(), 0);
    if (order == 1) std::reverse(turn.begin(), turn.end());
    for (int barriers = 0; barriers < 1000; ++barriers) {
        if (order > 1) std::shuffle(turn.begin(), turn.end(), rng);
        bool left = false;
        for (int w : turn) {
            for (bool ran = true; ran;) {
                ran = false;
                for (int i = w * kLanes; i < (w + 1) * kLanes; ++i)
                    if (lanes[i].state == Lane::kRuns) {
                        ran = true, current = i, threadIdx.x = i;
                        swapcontext(&scheduler, &lanes[i].context);
                    }
            }
        }
        for (Lane& l : lanes)
            if (l.state == Lane::kAtBarrier) l.state = Lane::kRuns, left = true;
            else if (l.state != Lane::kDone) return -1;  // lanes of a wave that wait for each other at different places
        if (!left) return barriers;
    }
    return -1;
}
