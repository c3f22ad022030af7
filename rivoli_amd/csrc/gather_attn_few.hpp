// Attention over an index list at d = 512 for calls of few workgroups (decode: one query): 16 heads a workgroup of
// eight waves, 64 slots at a time.
//
// What bounds it: the chain launch -> list entry -> row -> scores -> softmax -> values -> store of a share of one or
// two such tiles, on a part of the chip. So everything that can be asked for at once is: all 64 rows of a tile
// (eight a wave) behind one round trip for the list, the query beside them. Each wave takes 16 slots and half the
// dims of the scores (8 products), and 64 columns of the values (16); between them the scores go
// through LDS, where every wave reads them all and works out the same weights, so the reference maximum needs no
// exchange of its own. A query of 640 slots and 64 heads takes 40 such workgroups instead of ten of 64 heads, each with a
// quarter of the query and of the results: 17.1 -> 10.1 us with the merge of its ten shares.
#pragma once
#include "attend_common.hpp"

namespace rk {

constexpr int kGfThreads = 512;
constexpr int kGfWaves = kGfThreads / kWave;
constexpr int kGfHeads = 16;
constexpr int kGfSlots = 64;                    // slots a tile
constexpr int kGfRowsPerWave = kGfSlots / kGfWaves;
constexpr int kGfScoreStride = kGfSlots + 4;    // f32 a head, 16 bytes of padding
constexpr int kGfQueryAt = kGfSlots * kGaRowBytes;
constexpr int kGfScoresAt = kGfQueryAt + 2 * kGfHeads * kGaRowBytes;
constexpr int kGfFlagAt = kGfScoresAt + 2 * kGfHeads * kGfScoreStride * 4;
constexpr int kGfSmemBytes = kGfFlagAt + kGfWaves * 4;
static_assert(kGfSmemBytes <= 160 * 1024, "one workgroup a compute unit");

template <int QSPLIT, int PSPLIT>
__global__ __launch_bounds__(kGfThreads) void gather_attn_few_kernel(const GatherAttnArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[kGfSmemBytes];
    const lds_ptr<uint8_t> rows = (lds_ptr<uint8_t>)smem;               // [64] rows of a tile, bf16
    const lds_ptr<uint8_t> query = rows + kGfQueryAt;                   // [2][16] heads: values, remainders
    const lds_ptr<float> scores = (lds_ptr<float>)(rows + kGfScoresAt); // [2 halves of the dims][16 heads][slots]
    const lds_ptr<int> flag = (lds_ptr<int>)(rows + kGfFlagAt);         // a wave's heads have remainders
    const size_t t = blockIdx.x;
    const int head0 = blockIdx.y * kGfHeads;
    const int split = blockIdx.z;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, n16 = lane & 15;
    const int* const ix = a.idxs + t * a.topk;
    const int all_tiles = (a.topk + kGaTile - 1) / kGaTile;            // the plan's shares are of 32-slot tiles
    const int first = kGaTile * (int)((long long)split * all_tiles / a.n_splits);
    const int end = min(a.topk, kGaTile * (int)((long long)(split + 1) * all_tiles / a.n_splits));

    // ---- everything that needs no list entry, then the first tile's rows
    auto fetch = [&](int base) { return ix[min(base + lane, a.topk - 1)]; };  // slot base + lane of the list
    int entry = fetch(first);
    f32x4 qv[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int head = head0 + 2 * wave + i;
        const f32x4* src = reinterpret_cast<const f32x4*>(a.q + (t * a.h + (head < a.h ? head : 0)) * kGaD);
        qv[i][0] = src[lane], qv[i][1] = src[64 + lane];  // a head past h reads head 0: its results go nowhere
    }
    f32x4 raw[kGfRowsPerWave][2];
    uint64_t live = 0;  // of the tile that `raw` holds, one bit a slot
    auto ask = [&](int base) {
        live = __builtin_amdgcn_ballot_w64(base + lane < end && (unsigned)entry < (unsigned)a.n_kv);
#pragma unroll
        for (int i = 0; i < kGfRowsPerWave; ++i) {
            const int slot = kGfRowsPerWave * wave + i;
            const int p = (live >> slot) & 1 ? __builtin_amdgcn_readlane(entry, slot) : 0;  // masked: row 0, staged as zeros
            const f32x4* src = reinterpret_cast<const f32x4*>(a.kv + (size_t)p * kGaD);
            raw[i][0] = src[lane], raw[i][1] = src[64 + lane];
        }
    };
    ask(first);
    // rows hold dims 4 l .. and 256 + 4 l .. side by side at 16 l, the query's likewise
    auto packed = [&](f32x4 x, f32x4 y) {
        return u32x4{pack_bf16x2(x.x, x.y), pack_bf16x2(x.z, x.w), pack_bf16x2(y.x, y.y), pack_bf16x2(y.z, y.w)};
    };
    {
        uint32_t any = 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const lds_ptr<uint8_t> at = query + row_of_slot(2 * wave + i) * kGaRowBytes + 16 * lane;
            *(lds_ptr<u32x4>)at = packed(qv[i][0], qv[i][1]);
            if (QSPLIT == 2) {
                f32x4 lo[2];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float x = qv[i][k >> 2][k & 3];
                    lo[k >> 2][k & 3] = x - (float)(__bf16)x;
                    any |= __float_as_uint(x) & 0xffffu;
                }
                *(lds_ptr<u32x4>)(at + kGfHeads * kGaRowBytes) = packed(lo[0], lo[1]);
            }
        }
        if (QSPLIT == 2) {
            const bool has = __builtin_amdgcn_ballot_w64(any != 0) != 0;
            if (lane == 0) flag[wave] = has;
        }
    }

    const int group = wave & 3, half = wave >> 2;  // of the scores: 16 slots, half the dims
    // K-step j, lane group g: the 8 dims at bytes 512 half + 256 (g & 1) + 32 j + 16 (g >> 1) of a row (no two of the sixteen
    // lanes that a 16-byte LDS read serves together meet in a bank)
    const int dims_at = 512 * half + 256 * (g & 1) + 16 * (g >> 1);
    f32x4 o[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = f32x4{0, 0, 0, 0};
    float m_ref = -INFINITY, l_sum = 0.0f;
    bf16x8 qh[8], ql[QSPLIT == 2 ? 8 : 1];
    bool has_lo = false, loaded = false;

    for (int base = first; base < end; base += kGfSlots) {
#pragma unroll
        for (int i = 0; i < kGfRowsPerWave; ++i) {
            const int slot = kGfRowsPerWave * wave + i;
            u32x4 v = packed(raw[i][0], raw[i][1]);
            if (!((live >> slot) & 1)) v = u32x4{0u, 0u, 0u, 0u};
            *(lds_ptr<u32x4>)(rows + ((slot & ~15) + row_of_slot(slot & 15)) * kGaRowBytes + 16 * lane) = v;
        }
        const uint64_t mine = live;
        if (base + kGfSlots < end) entry = fetch(base + kGfSlots);
        __syncthreads();
        if (!loaded) {
            loaded = true;
            const lds_ptr<uint8_t> at = query + row_of_slot(n16) * kGaRowBytes + dims_at;
#pragma unroll
            for (int j = 0; j < 8; ++j) qh[j] = *(lds_ptr<bf16x8>)(at + 32 * j);
            if (QSPLIT == 2) {
                int any = 0;
#pragma unroll
                for (int w = 0; w < kGfWaves; ++w) any |= flag[w];
                has_lo = __builtin_amdgcn_readfirstlane(any) != 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) ql[j] = *(lds_ptr<bf16x8>)(at + kGfHeads * kGaRowBytes + 32 * j);
            }
        }
        // ---- S^T[slot][head]: 16 slots, half the dims; a query that is bf16-valued has no remainder's products
        f32x4 s = {0, 0, 0, 0};
        {
            const lds_ptr<uint8_t> at = rows + (16 * group + row_of_slot(n16)) * kGaRowBytes + dims_at;
            bf16x8 k[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) k[j] = *(lds_ptr<bf16x8>)(at + 32 * j);
#pragma unroll
            for (int j = 0; j < 8; ++j) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j], qh[j], s, 0, 0, 0);
            if (QSPLIT == 2 && has_lo) {
#pragma unroll
                for (int j = 0; j < 8; ++j) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j], ql[j], s, 0, 0, 0);
            }
        }
        *(lds_ptr<f32x4>)(scores + (half * kGfHeads + n16) * kGfScoreStride + 16 * group + 4 * g) = s;
        if (base + kGfSlots < end) ask(base + kGfSlots);
        // the values' operands: four slots of column n16 a read, as in gather_attn_d512
        const lds_ptr<uint8_t> vrow = rows + row_of_slot(4 * g + (n16 >> 2)) * kGaRowBytes + (64 * wave + 4 * (n16 & 3)) * 2;
        bf16x8 v[2][4];
#pragma unroll
        for (int tile = 0; tile < 2; ++tile)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                typedef short s16x4 __attribute__((ext_vector_type(4)));
                typedef short s16x8 __attribute__((ext_vector_type(8)));
                const lds_ptr<uint8_t> at = vrow + 32 * tile * kGaRowBytes + 32 * c;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<s16x4>)at);
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr<s16x4>)(at + 16 * kGaRowBytes));
                const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                v[tile][c] = __builtin_bit_cast(bf16x8, both);
            }
        __syncthreads();
        // ---- softmax, in every wave the same: the lane's 16 slots of head n16
        float x[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // slots 16 q + 4 g ..
            const lds_ptr<float> at = scores + n16 * kGfScoreStride + 16 * q + 4 * g;
            const f32x4 s0 = *(lds_ptr<f32x4>)at, s1 = *(lds_ptr<f32x4>)(at + kGfHeads * kGfScoreStride);
            const uint32_t bits = (uint32_t)(mine >> (16 * q)) >> (4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * q + i] = (bits >> i) & 1 ? (s0[i] + s1[i]) * a.qscale : -INFINITY;
        }
        float top = x[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) top = fmaxf(top, x[i]);
        top = fmaxf(rows_max(top), m_ref);
        const float mu = top == -INFINITY ? 0.0f : top;
        const float corr = m_ref == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_ref - mu);
        m_ref = top;
        l_sum *= corr;
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] *= corr;
        // the weights as the value products' B operand: 8 slots of a 32-slot tile, rounded and their remainders;
        // carried once (PSPLIT 1), the denominator sums the rounded ones
        bf16x8 p[2], p_lo[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float e = __builtin_amdgcn_exp2f(x[i] - mu);  // masked -> 0
            const __bf16 w = (__bf16)e;
            p[i >> 3][i & 7] = w;
            if (PSPLIT == 2) p_lo[i >> 3][i & 7] = (__bf16)(e - (float)w);
            l_sum += PSPLIT == 2 ? e : (float)w;
        }
#pragma unroll
        for (int tile = 0; tile < 2; ++tile)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                o[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[tile][c], p[tile], o[c], 0, 0, 0);
                if (PSPLIT == 2) o[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[tile][c], p_lo[tile], o[c], 0, 0, 0);
            }
    }

    // ---- O^T: the lane has columns 64 wave + 16 c + 4 g .. of head n16, which are dims 4 (8 wave + 2 c + (g >> 1)) + 256 (g & 1) ..
    l_sum = rows_sum(l_sum);
    const int head = head0 + n16;
    if (head >= a.h) return;
    const int dim = 4 * (8 * wave + (g >> 1)) + 256 * (g & 1);
    if (a.n_splits > 1) {  // a share of the list: unnormalised sums and (m, l) for the combine kernel
        const size_t rec = (t * a.n_splits + split) * a.h + head;
#pragma unroll
        for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4*>(a.part_acc + rec * kGaD + dim + 8 * c) = o[c];
        if (wave == 0 && g == 0) a.part_ml[rec * 2] = m_ref, a.part_ml[rec * 2 + 1] = l_sum;
        return;
    }
    // nothing live: m_ref is still -inf and the query's output is NaN
    const float l = m_ref == -INFINITY ? NAN : l_sum + exp2f(a.sink[head] * kLog2e - m_ref);
    const float l_inv = 1.0f / l;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        f32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = (float)(__bf16)(o[c][i] * l_inv);
        *reinterpret_cast<f32x4*>(a.o + (t * a.h + head) * kGaD + dim + 8 * c) = r;
    }
}

}  // namespace rk
