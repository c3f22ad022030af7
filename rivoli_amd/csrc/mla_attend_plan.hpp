// Which kernel an MLA attention call takes and how its 32-token tiles become work items: host
// arithmetic on the call's shape alone (no length is known there), shared by the launchers of
// mla_attend.hip and the tests that hold the rules.
#pragma once

namespace rk {

constexpr int kTile = 32;                  // tokens per tile
constexpr int kAttTargetGroups = 256;      // one workgroup per CU of a 256-CU part
constexpr int kAttDies = 8;                // workgroups are dealt to the dies in turn
constexpr int kAttMinTilesPerSplit = 8;    // below 256 rows a split costs more than it buys
constexpr int kAttMaxSplits = 64;
constexpr int kRefMaxSplits = 16;          // what rivoli_mla_attend_scratch_floats prices (attn.hip:66,98-103)
constexpr int kDealMaxSeqs = 1024;         // dealing keeps a prefix sum over the sequences in LDS
constexpr int kH16Heads = 16;              // mla_attend_heads16.hpp: heads and waves of a workgroup
constexpr int kH16Waves = 4;
constexpr int kH16WholeTiles = 32;         // past these a whole sequence is a workgroup's for too long
constexpr int kSeqDealMax = 64;            // SeqDeal: sequences, one a lane
constexpr int kSeqDealMaxTiles = 1 << 19;  // of a sequence: its quotients stay under 2^24

// Work plan of the workgroups of 64 heads. `n_splits` is a pure function of the call's shape; with
// more than one split the attended rows of ALL sequences, in tiles, are dealt evenly to n_seqs *
// n_splits work items from the device-side lengths (a work item may cover parts of several
// sequences, a sequence several work items), so ragged batches keep every CU busy.
struct AttendPlan {
    int n_splits;
    int n_items;    // work items per head block when dealing (0 = one workgroup per sequence)
    int n_records;  // partial records when dealing: a (work item, sequence) pair is item + seq
};

static inline AttendPlan attend_plan(int n_seqs, int H, int max_rows) {
    const int head_blocks = (H + 63) / 64;
    const int tiles = (max_rows + kTile - 1) / kTile;
    const long long per_split = (long long)n_seqs * head_blocks;
    int by_grid = (int)((kAttTargetGroups + per_split - 1) / per_split);
    int by_work = tiles / kAttMinTilesPerSplit;
    int n = by_grid < by_work ? by_grid : by_work;
    if (n > kAttMaxSplits) n = kAttMaxSplits;
    if (n < 1 || n_seqs > kDealMaxSeqs) n = 1;
    AttendPlan p;
    p.n_splits = n;
    p.n_items = n > 1 ? n * n_seqs : 0;
    p.n_records = n > 1 ? p.n_items + n_seqs : 0;
    return p;
}

// The same for the linear slabs' one sequence, cut to what the caller's scratch holds: `fit` records of
// which one is spare. Up to 512 heads, where its workgroups have 16 of them (heads16_pays), a call that is cut at
// all is cut to 128 rows a work item, where the paged workgroups of 64 heads want 256: 64 heads, 512 rows 16.3 -> 13.1 us, 1 024
// 16.5 -> 13.3, 1 800 20.0 -> 16.8; 256 rows are not worth a second launch, and past 2 500 the scratch decides. The general form,
// which takes other widths and slabs off a 16-byte boundary, gains as much: 64 heads of width 256, 512 rows 43.4 -> 31.5,
// 1 024 43.4 -> 34.4, 1 800 45.9 -> 45.6; 384 47.0 -> 35.3, 47.2 -> 35.5, 49.7 -> 41.7; 512 from 8 bytes on 50.9 -> 38.8, 51.1 -> 39.1, 53.3 -> 42.4.
static inline AttendPlan linear_plan(int H, int nr, int fit, bool scratch) {
    AttendPlan p = attend_plan(1, H, nr);
    if (p.n_splits > 1 && H <= kH16Heads * kAttTargetGroups / kAttDies) p.n_splits = (nr + kTile - 1) / kTile / kH16Waves;
    if (p.n_splits > fit - 1) p.n_splits = fit - 1;
    if (!scratch || p.n_splits < 2) p.n_splits = 1;
    p.n_items = p.n_splits > 1 ? p.n_splits : 0;
    p.n_records = p.n_items ? p.n_items + 1 : 0;
    return p;
}

// Rounds of workgroups a die's 32 compute units take for `items` work items: the head groups of an
// item sit on one die (mla_attend_heads16_kernel).
constexpr int kAttDieUnits = kAttTargetGroups / kAttDies;
static inline long long heads16_rounds(long long items, long long groups) {
    const long long per_die = (items + kAttDies - 1) / kAttDies * groups;
    return (per_die + kAttDieUnits - 1) / kAttDieUnits;
}

// The work items of a call by 16 heads a workgroup: one workgroup per compute unit, at least a tile
// per wave, and no more partial records than `plan` (which the caller's scratch was sized by) has.
// A die takes whole items, so three groups of heads make 8 x 10 items, not 85: with 85 five of the
// dies had 33 workgroups for their 32 units and the call two rounds (21 x 1 600 tokens 50 us, with 80
// 33; 112 heads, 5 x 4 000 55 and 36).
// Up to 64 sequences no work item meets two of them, so their number need not be a multiple of the
// sequences'; more sequences, or longer ones than SeqDeal counts, share the tiles evenly. Fewer than
// two work items a sequence are not worth the merge, but for one thing: up to 16 heads a call has
// nowhere else to go, and one long sequence must not keep a workgroup to itself. Past 32 tiles a work
// item a sequence shares those batches' tiles too: 200 sequences, one of 32 768 tokens and the others
// of 100, 769 -> 72 us (one of 4 096 106 -> 36; all of 4 096 111 -> 118, the merge's launch).
static inline AttendPlan heads16_plan(const AttendPlan& plan, int n_seqs, int H, int max_rows, bool& by_seq) {
    const int tiles = max_rows / kTile + (max_rows % kTile != 0);
    const int groups = (H + kH16Heads - 1) / kH16Heads;
    const long long most = (long long)n_seqs * (tiles / kH16Waves);
    by_seq = n_seqs <= kSeqDealMax && tiles <= kSeqDealMaxTiles;
    long long n = groups <= kAttDieUnits ? kAttDieUnits / groups * kAttDies : kAttTargetGroups / groups;
    if (n > most) n = most;
    if (n > plan.n_items) n = plan.n_items;
    if (!by_seq) n = n / n_seqs * n_seqs;
    const int least = groups == 1 && tiles > kH16WholeTiles ? n_seqs : 2 * n_seqs;
    if (n < least) n = 0, by_seq = false;
    AttendPlan p;
    p.n_items = (int)n;
    p.n_splits = n ? (int)((n + n_seqs - 1) / n_seqs) : 1;
    p.n_records = n ? p.n_items + n_seqs : 0;
    return p;
}

// Whether a call goes to the workgroups of 16 heads: its 32-token tiles times its groups of 16
// heads, before the lengths are known. (The figures of this side here and below are those of a tile a wave;
// eight waves on a tile, heads16_few, take 2 to 50 % off them.) Parity mode, 64 heads: 1 x 4 096 tokens (512) 21.5 us
// against 34.5 in workgroups of 64 heads, 32 x 1 000 (4 096) 33 against 39, 6 ragged of up
// to 9 000 (6 768) 39 against 51 with the append, 32 listed sets of 2 048 rows (8 192) 45 against 48, 32 x 4 096 (16 384) 73 against 64.
// The 8-bit modes' kernel is the faster one sooner: 8 listed sets of 2 048 rows (2 048) 24 us in
// the parity mode here against 34 at precise 4, 32 x 1 000 (4 096) 32 against 33, 32 listed sets
// (8 192) 44 against 42; below the line they run in the parity mode. Up to 16 heads the other
// kernels' workgroups are three quarters empty: 32 x 16 384 tokens 84 us against 163 (precise 2)
// and 107 (4).
constexpr long long kH16MaxWork = 8192, kH16MaxWork8Bit = 4096;
// Above that line, dense calls of few enough sequences for SeqDeal to cut them well (two and a half
// work items a sequence; at 2, 32 x 2 989 ragged tokens 57 us against 52) still go there while the
// workgroups of 64 heads would need a second, nearly empty round: they are dealt as ceil(256 / per
// split) splits, so 18 sequences are 270 workgroups for 256 compute units. Ragged, parity mode: 7 x
// 11 360 tokens 38 us against 64, 17 x 10 161 (21 624) 63 against 83, 11 x 12 613 of 128 heads
// (34 760) 178 against 174; precise 4: 13 x 7 584 (12 324) 41 against 66, 17 x 7 255 (15 436) 57
// against 69, 18 x 10 262 (23 112) 107 against 102. Calls that those workgroups fill in one round
// change sides sooner: 8 x 11 058 (11 072) 49 against 52, 4 x 32 768 (16 384) 74 against 71; precise
// 4: 1 x 32 768 (4 096) 43 against 51, 4 x 32 768 70 against 59.
// Neither line holds for the linear slabs: their other kernel is the general form of the 64-head one and
// their scratch gives it 15 work items. 64 heads: 512 rows 19 us against 50, 65 536 rows 139 against 484,
// 200 000 rows 385 against 1 420; 512 heads, 20 000 rows 92 against 172.
constexpr long long kH16MaxWorkFull = 12288, kH16MaxWorkFull8Bit = 8192;
constexpr long long kH16MaxWorkSpill = 24576, kH16MaxWorkSpill8Bit = 16384;
// Calls whose sequences stay whole (one workgroup a sequence and head group) go there while that
// takes no more rounds of workgroups than a workgroup a sequence and 64 heads does. A round costs 11
// us and 2.6 per four tiles here, 7 us and 2.4 per tile there: 128 heads, parity mode, 32 x 128
// tokens 13 us against 19, 64 x 128 (two rounds) 23 against 21, 128 x 128 (four) 45 against 24; 64
// heads, 256 x 256 tokens 59 against 34; precise 4, 128 x 256 tokens 32 against 22. Two rounds are
// still the faster at 15 to 20 tiles (64 x 512 tokens of 128 heads 44 against 50, ragged 41 against
// 56; 15 tiles 43 against 44, ragged 40 against 41; 10 tiles 36 against 33), where the other kernel
// starts to split and merge, and past them (34 x 960 tokens 67 against 49) where its splits are more
// than a round themselves (32 heads, 136 x 960 tokens 67 against 93). One tile, two of up to 16
// heads and two dense ones of up to 32 leave half the waves and more without any: 16 heads, 32 tokens
// 11 us against 8, 64 tokens 11.0 against 10.0; 64 heads, one token 12.7 against 10.8, 32 tokens 11.0
// against 11.0. Three tiles of more than a round of sequences are worth it where all are as long, and not
// in a ragged batch (8 heads, 257 sequences, even 20 against 23, lengths to 96 from 3 on 21 against 18, one
// of 96 among 6s 21 against 14; four tiles 20 against 28, 22 against 20 and 21 against 14; in one round 11
// against 13, 12.4 against 12.3 and 12.2 against 11.8). (The 8-bit kernel is not faster there, 12 us
// against 16, nor is the general form of the linear slabs, 10.9 against 24.8.) Past 32 tiles the call lasts as long as its longest sequence
// in one workgroup, and the other kernel deals them out: 64 heads, 33 x 1 984 tokens 60 us against 46,
// one of 1 984 among 32 of 100 58 against 36; unless its splits, again, are more than a round (32
// heads, 80 x 1 600 tokens 50 against 80).
constexpr int kH16TwoRoundTiles = 15, kH16TwoRoundMaxTiles = 20;
static inline bool heads16_whole_pays(const AttendPlan& plan, int n_seqs, int H, int tiles, bool f8, bool dense,
                                      bool linear) {
    const int few = H <= 16 && n_seqs > kAttTargetGroups ? 3 : H <= 16 || (dense && H <= 32) ? 2 : 1;
    if (!f8 && !linear && tiles <= few) return false;
    const long long blocks = (H + 63) / 64;
    const bool spills = plan.n_items * blocks > kAttTargetGroups;
    if (!linear && H > kH16Heads && tiles > kH16WholeTiles) return spills;
    const long long rounds = heads16_rounds(n_seqs, (H + kH16Heads - 1) / kH16Heads);
    if (rounds <= (n_seqs * blocks + kAttTargetGroups - 1) / kAttTargetGroups) return true;
    return !f8 && rounds == 2 && tiles >= kH16TwoRoundTiles && (tiles <= kH16TwoRoundMaxTiles || spills);
}
// The head groups of a work item are a die's 32 units at most, or the item takes rounds of its own: past
// 512 heads calls stay with the other kernel (2 048 heads, parity mode, 1 024 listed rows 92 us here
// against 44; 768 dense, 1 638 rows 44 against 40, precise 3, 857 rows 43 against 31; 520 with two
// sequences listed 34 against 40). The general form of the linear slabs is slower than that kernel: 1 024
// heads 512 rows 36 us here against 53, 2 048 rows 53 against 60, 4 096 rows 82 against 68; 1 536 heads 1 024
// rows 75 against 59, 2 048 heads 2 048 rows 153 against 67.
constexpr int kH16ManyHeadsTiles = 64;  // linear slabs, up to two rounds of head groups
// `cut`: heads16_plan shares the sequences among work items.
static inline bool heads16_pays(const AttendPlan& plan, bool cut, int n_seqs, int H, int max_rows, int precise,
                                bool dense, bool linear) {
    const long long groups = (H + kH16Heads - 1) / kH16Heads;
    const int tiles = max_rows / kTile + (max_rows % kTile != 0);
    const long long work = (long long)n_seqs * tiles * groups;
    const bool f8 = precise > 2;
    if (!cut && !heads16_whole_pays(plan, n_seqs, H, tiles, f8, dense, linear)) return false;
    if (groups > kAttDieUnits && !(linear && groups <= 2 * kAttDieUnits && tiles <= kH16ManyHeadsTiles)) return false;
    if (linear || groups == 1 || work <= (f8 ? kH16MaxWork8Bit : kH16MaxWork)) return true;
    if (!dense || 5 * n_seqs * groups > 2 * kAttTargetGroups) return false;
    const bool spills = (long long)plan.n_items * ((H + 63) / 64) > kAttTargetGroups;
    return work <= (spills ? (f8 ? kH16MaxWorkSpill8Bit : kH16MaxWorkSpill) : (f8 ? kH16MaxWorkFull8Bit : kH16MaxWorkFull));
}

// Which kernel the workgroups of 16 heads run. Eight waves on a tile of 64 tokens (mla_attend_few.hpp) are the faster in
// every shape tried that has three groups of heads and more, linear slabs or short work items: linear, 64 heads, 33 rows
// 12.6 -> 7.1 us, 300 rows 19.4 -> 13.7, 8 192 rows 31.4 -> 28.1, 300 000 rows 564 -> 524; 20 x 9 000 tokens of 64 heads 94.5 -> 90.1.
// One or two groups of heads that walk long work items have each row from memory and wait for it; a
// tile of its own per wave (mla_attend_heads16.hpp) keeps more of them on their way. Parity mode, 16 heads, per tile-a-wave
// and eight waves: dense, one sequence of 100 000 tokens (49 tiles a work item) 64.4 us and 63.1, 300 000 (146) 138.5 and 139.1,
// 800 000 (390) 325 and 340. Work items that fill the chip and cover their sequences from end to end reach that sooner, the more
// so the more even the batch: whole sequences, 256 of 1 500 (47) 56.7 and 55.1, of 2 000 (63) 75.6 and 76.2 (of one head 69.9 and 74.4; ragged 66.0 and 63.6),
// of 3 000 (94) 107.8 and 109.8 (88.2 and 90.7); shared evenly, 192 of 3 000 (94) 100.5 and 99.9 (87.5 and 76.7), of 4 000 (125) 124.7
// and 128.4 (104.1 and 91.9). Lists, whose rows are scattered, sooner too: 64 of 6 000 rows (47) 68 and 66, 300 of 3 000 (94)
// 180 and 186, 257 of 6 000 (188) 323 and 355. With q and weights in one term (precise 0) cut dense sequences: 100 000 tokens (49) 57.6
// and 57.7, 200 000 (98) 88.7 and 91.4; whole ones 257 of 3 000 (94) 158.0 and 156.4, of 4 000 (125) 195.4 and 201.3.
constexpr int kFewMaxTiles = 128, kFewMaxTilesShared = 96, kFewMaxTilesWhole = 56, kFewMaxTilesListed = 48;  // of a work item
constexpr int kFewMaxTilesOneTerm = 64, kFewMaxTilesOneTermWhole = 96;
static inline bool heads16_few(const AttendPlan& p, bool by_seq, int n_seqs, int H, int max_rows, int precise, bool dense,
                               bool linear) {
    if (linear || H > 2 * kH16Heads) return true;
    const long long tiles = max_rows / kTile + (max_rows % kTile != 0);
    const long long longest = p.n_items ? (n_seqs * tiles + p.n_items - 1) / p.n_items : tiles;
    if (!dense) return longest <= kFewMaxTilesListed;
    if (precise == 0) return longest <= (p.n_items ? kFewMaxTilesOneTerm : kFewMaxTilesOneTermWhole);
    return longest <= (by_seq ? kFewMaxTiles : p.n_items ? kFewMaxTilesShared : kFewMaxTilesWhole);
}

// A call of the shipped row widths whose rows are whole 16-byte pieces. `plan`: attend_plan's or
// linear_plan's.
struct AttendRoute {
    bool heads16;  // workgroups of 16 heads; else of 64
    bool by_seq;   // no work item has tiles of two sequences (SeqDeal)
    bool few;      // eight waves on a tile, else a tile a wave
    AttendPlan plan;
};
static inline AttendRoute attend_route(const AttendPlan& plan, int n_seqs, int H, int max_rows, int precise, bool dense,
                                       bool linear) {
    bool by_seq;
    const AttendPlan p = heads16_plan(plan, n_seqs, H, max_rows, by_seq);
    if (!heads16_pays(plan, p.n_items > 0, n_seqs, H, max_rows, precise, dense, linear)) return {false, false, false, plan};
    return {true, by_seq, heads16_few(p, by_seq, n_seqs, H, max_rows, precise, dense, linear), p};
}

// Workgroups of 32 heads (mla_attend_heads32.hpp) for calls that SeqDeal cuts: one a compute unit again, a die taking whole work
// items, and no more partial records than `plan` has. n_items 0: not such a call.
constexpr int kWideHeads = 32;
constexpr int kWideRun = 2;  // SeqDeal's unit there: a tile of 64 tokens
static inline AttendPlan heads32_plan(const AttendPlan& plan, int n_seqs, int H, int max_rows) {
    const long long tiles = max_rows / kTile + (max_rows % kTile != 0);
    const int groups = (H + kWideHeads - 1) / kWideHeads;
    AttendPlan p = {1, 0, 0};
    if (n_seqs > kSeqDealMax || tiles > kSeqDealMaxTiles || groups > kAttDieUnits || H <= kH16Heads) return p;
    long long n = kAttDieUnits / groups * kAttDies;
    const long long most = n_seqs * (tiles / kWideRun);
    if (n > most) n = most;
    if (n > plan.n_items) n = plan.n_items;
    if (n < 2 * n_seqs) return p;
    p.n_items = (int)n, p.n_splits = (int)((n + n_seqs - 1) / n_seqs), p.n_records = p.n_items + n_seqs;
    return p;
}
// Whether such a call goes there; `heads16`: it would go to workgroups of 16 heads otherwise, else to those of 64. us, parity mode unless
// said, there -> here. A tile of 32 heads costs about two of 16, and a work item 1 us more, so from 16 heads it is the finer cut of
// a batch that pays, half as many groups making twice the work items: listed sets of 2 048 rows, 12 of 128 heads (work 6 144) 41.5 -> 37.6,
// 32 of 64 (8 192) 44.6 -> 42.3, but 16 of 64 (4 096) 28.1 -> 30.5; dense, 17 x 7 255 ragged at precise 4 (15 436) 46.5 -> 42.5, 7 x 11 360 ragged (9 968)
// 39.5 -> 39.2, but 20 x 3 000 ragged (7 520) 31.4 -> 32.0 and 6 x 9 000 (6 768) 34.3 -> 35.5.
// From 64 heads: calls that those would need a second, nearly empty round for, 24 x 8 000 117 -> 77, 9 x 16 384 of 128 heads ragged 130 -> 75, 48 listed
// sets of 2 048 rows 87 -> 66, and at precise 4 18 x 10 262 ragged 72 -> 51, 11 x 12 613 of 128 heads 96 -> 66; in one round up to 24 576: 32 x 6 000
// (24 064) 79.1 -> 78.9, ragged 63 -> 57, 32 x 4 096 at precise 0 (16 384) 58 -> 51, but 16 x 16 384 (32 768) 94 -> 97, and the 8-bit kernel stays the faster.
// Up to 32 heads those workgroups are half empty.
// What a call takes lies on a line over its longest work item, in tiles of an even batch (a thousand calls of 17 to 1 024 heads, most within
// 3 %): here 19.5 us and 2.25 per tile of 64 tokens; by 16 heads 15.6 and 1.5; by 64 in two rounds, per tile of 32 in both of them,
// 35 and 2.0 in the parity mode, of listed rows 44 and 1.9, but with the 8-bit instructions 43 and 1.05 (precise 3: 38 and 0.96), listed 34 and 1.7. So a
// second round of the 8-bit kernel's is the shorter way past a length, and such calls stay there: even, precise 4, 27 x 16 384 of 128 heads 277 against 316 here, 24 x
// 12 000 of 112 175 and 232, 6 x 16 384 of 384 175 and 304, 3 x 24 000 of 640 221 and 440, but 17 x 9 000 of 64 85 and 67, 12 x 6 000 of 128 85 and 63. Ragged
// batches gain sooner, the more so the more sequences (22 x 6 000 of 128 heads even 112 and 124, ragged 94 and 72): the line lies between the
// two; 17 x 13 000 of 128 heads still come here (even 0.89 of the speed, ragged 1.21), 24 x 13 000 do not (0.74 and 0.95). In the parity mode
// only head counts that leave compute units out come to it: 3 x 16 384 of 640 268 and 304.
// Lists whose work items come out no more than half as long again by 16 heads stay with those: 3 of 8 192 rows of 128 heads 0.94 of the speed here, 12 of
// 4 096 of 80 0.93, 9 of 8 192 of 33 0.94. So do lists that 64 heads take in one full round of up to four work items a
// sequence: 64 of 2 048 rows of 64 heads 0.88 of the speed, 32 of 128 heads 0.97; of eight, 16 of 4 096 of 128 heads, 1.03.
constexpr long long kWideMinWork = 8192, kWideMinWorkListed = 5120, kWideMaxWork = 24576;
constexpr int kWideMinSplitsListed = 5;
// Tiles of the longest of `items` work items of an even batch that SeqDeal cuts.
static inline long long seq_deal_run(long long tiles, int n_seqs, int items) {
    const int each = items / n_seqs;
    return (tiles + each - 1) / each;
}
static inline bool heads32_pays(const AttendPlan& p, const AttendPlan& plan, const AttendRoute& route, int n_seqs, int H, int max_rows,
                                int precise, bool dense) {
    const long long tiles = max_rows / kTile + (max_rows % kTile != 0);
    const long long run = (seq_deal_run(tiles, n_seqs, p.n_items) + kWideRun - 1) / kWideRun;  // tiles of 64 tokens
    if (route.heads16) {
        const long long run16 = (seq_deal_run(tiles, n_seqs, route.plan.n_items) + kWideRun - 1) / kWideRun;
        if (!dense && precise > 0 && 2 * run16 < 3 * run + 6) return false;
        return n_seqs * tiles * ((H + kH16Heads - 1) / kH16Heads) > (dense ? kWideMinWork : kWideMinWorkListed);
    }
    const int groups = (H + kWideHeads - 1) / kWideHeads;
    const long long there = (long long)plan.n_items * ((H + 63) / 64);
    if (there > kAttTargetGroups) {
        if (precise == 0) return true;
        const long long rounds = (there + kAttTargetGroups - 1) / kAttTargetGroups;
        const long long run64 = rounds * n_seqs * tiles / plan.n_items;
        if (precise > 2) return 100 * run <= (dense ? 47 * run64 + (n_seqs < 8 ? 1400 : 2200) : 69 * run64 + 600);
        return 100 * run <= (dense ? 90 * run64 + 1200 : 64 * run64 + 1400);
    }
    if (precise > 2 || 4 * p.n_items * groups < 3 * kAttTargetGroups) return false;
    if (groups == 1) return true;
    if (!dense && (precise == 2 || (precise == 1 && groups == 2)) && plan.n_splits < kWideMinSplitsListed && there == kAttTargetGroups) return false;
    return n_seqs * tiles * 2 * groups <= kWideMaxWork;
}
// A paged call's work items there, n_items 0 where `route`, attend_route's, stands.
static inline AttendPlan heads32_route(const AttendPlan& plan, const AttendRoute& route, int n_seqs, int H, int max_rows, int precise,
                                       bool dense) {
    AttendPlan p = heads32_plan(plan, n_seqs, H, max_rows);
    // (sequences that stay whole, or that one long one of many must not keep a workgroup with, stay where they are)
    if (!p.n_items || (route.heads16 && !route.by_seq) || !heads32_pays(p, plan, route, n_seqs, H, max_rows, precise, dense)) p.n_items = 0;
    return p;
}

}  // namespace rk
