// Which kernel a call of the block scorer takes (head dim 128, up to 64 heads, kv on 16 bytes) and its share of the blocks: host
// arithmetic on the call's shape alone, shared by the launcher of block_index.hip and the tests that hold the rule.
#pragma once

namespace rk {

constexpr int kPairQueries = 8;      // of a workgroup of the many-query kernels: four waves of two
constexpr int kPairTile = 32;        // blocks of a matrix tile
constexpr int kPairSplitMax = 4096;  // blocks of a split: one bit of a 128-bit mask per tile
// Up to here a workgroup per (query, 64 blocks) is the faster: 4 queries x 4 096 blocks 7 us against
// 10 (4 x 8 192, 512 workgroups: 11.3 against 10.4; 300 queries x 75, 600: 15 against 10). One query
// has no second for the many-query kernel's wave: 65 536 blocks 18 us against 25.
constexpr int kOneGroups = 384;
// Workgroups of so many blocks turn their q rows into fp4 codes, which takes a wave 2 200 vector instructions where bf16 operands
// take 900: 192 blocks (2 049 x 512) 37.5 us as bf16 and 33.5 so, 384 (3 000 x 750) 54 and 46; 128 (1 500 x 375) 26.6 and 26.2, 64 (700 x 175)
// 10.4 and 11.5. Rows that are exact but no codes pay for finding that out: 8 192 queries of such q 229 -> 234, of such kv 208 -> 217, 2 049 38 -> 42
// and 37 -> 41.
constexpr int kFp4Blocks = 192;

enum class ScoreKernel { kOne32, kOne64, kPair, kCodes, kNone };  // a workgroup per query and 32 or 64 blocks; many queries; neither
struct ScorePlan {
    ScoreKernel kernel;
    int split;              // blocks of a workgroup of the many-query kernels
    unsigned groups, rows;  // their grid: query groups, splits
};
static inline ScorePlan score_plan(int s, int n_comp) {
    const long long groups = ((long long)n_comp + 63) / 64;
    // half the blocks a workgroup while there is a compute unit for each (8 192 blocks 6.1 us, 7.1 in
    // 64s; 16 384 blocks 7.1 us in 64s, 8.5 in 32s)
    if (s == 1 || s * groups <= kOneGroups) return {s * 2 * groups <= 256 ? ScoreKernel::kOne32 : ScoreKernel::kOne64, 0, 0, 0};
    // two workgroups per compute unit at a time; splits of the blocks while the queries alone
    // give fewer than two rounds of those (a split reads its queries' rows again)
    const unsigned t_groups = (unsigned)(((long long)s + kPairQueries - 1) / kPairQueries);
    const long long tiles = ((long long)n_comp + kPairTile - 1) / kPairTile;
    long long splits = t_groups >= 1024 ? 1 : 1024 / t_groups;
    if (splits > groups) splits = groups;
    int per = (int)((groups + splits - 1) / splits) * 64;
    const bool codes = per >= kFp4Blocks;
    // A tile each where that leaves compute units over, or is still one round and the q rows (32 KB
    // a query) stay in a die's 4 MB of cache, which every one of a query's workgroups reads them
    // through: 300 x 75 (114 workgroups) 11.7 -> 10.5 us, 5 x 8 192 (256) 10.1 -> 8.8; but 150 x 300 (190,
    // 4.9 MB) 10.1 -> 11.9.
    if (t_groups * tiles <= 128 || (t_groups * tiles <= 256 && t_groups <= 13)) per = kPairTile;
    if (per > kPairSplitMax) per = kPairSplitMax;
    const unsigned rows = (unsigned)(((long long)n_comp + per - 1) / per);
    return {rows > 65535u ? ScoreKernel::kNone : codes ? ScoreKernel::kCodes : ScoreKernel::kPair, per, t_groups, rows};
}

}  // namespace rk
