// The launchers' routing rules (rivoli_amd/csrc/mla_attend_plan.hpp, gather_attn_plan.hpp, block_index_plan.hpp) as C functions.
#include "../../rivoli_amd/csrc/block_index_plan.hpp"
#include "../../rivoli_amd/csrc/gather_attn_plan.hpp"
#include "../../rivoli_amd/csrc/mla_attend_plan.hpp"

// 1: workgroups of 16 heads, 0: of 64. out: items, by_seq, records of the route; items, records the
// caller's scratch is sized by; whether eight waves share a tile. linear: 0 a paged call, 1 the linear slabs with scratch, 2 without.
extern "C" int attend_route(int n_seqs, int H, int max_rows, int precise, int listed, int linear, int out[6]) {
    const rk::AttendPlan plan = linear ? rk::linear_plan(H, max_rows, rk::kRefMaxSplits, linear == 1)
                                       : rk::attend_plan(n_seqs, H, max_rows);
    const rk::AttendRoute r = rk::attend_route(plan, n_seqs, H, max_rows, precise, !listed && !linear, linear != 0);
    out[0] = r.plan.n_items, out[1] = r.by_seq, out[2] = r.plan.n_records;
    out[3] = plan.n_items, out[4] = plan.n_records, out[5] = r.few;
    return r.heads16;
}

// The same call's work items in workgroups of 32 heads, 0 where it stays with attend_route's.
extern "C" int attend_wide_items(int n_seqs, int H, int max_rows, int precise, int listed) {
    const rk::AttendPlan plan = rk::attend_plan(n_seqs, H, max_rows);
    const rk::AttendRoute r = rk::attend_route(plan, n_seqs, H, max_rows, precise, !listed, false);
    return rk::heads32_route(plan, r, n_seqs, H, max_rows, precise, !listed).n_items;
}

extern "C" long long marked_block(unsigned row, unsigned group) { return rk::marked_block(row, group); }

// 0 and 1: a workgroup per query and 32 or 64 blocks; 2: many queries, bf16; 3: fp4 codes; 4: neither. out: blocks of a workgroup, the grid.
extern "C" int score_plan(int s, int n_comp, int out[3]) {
    const rk::ScorePlan p = rk::score_plan(s, n_comp);
    out[0] = p.split, out[1] = (int)p.groups, out[2] = (int)p.rows;
    return (int)p.kernel;
}
