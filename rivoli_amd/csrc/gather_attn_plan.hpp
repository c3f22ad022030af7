// Which workgroup of the index-list attention's second pass has which block (a query's 64 heads): integer arithmetic shared
// by gather_attn.hip and the test that holds it.
#pragma once

#if defined(__HIP__)
#define RK_BOTH __host__ __device__
#else
#define RK_BOTH
#endif

namespace rk {

constexpr int kGaTargetGroups = 256;  // one workgroup per CU of a 256-CU part

// A group's block in row `row` of kGaTargetGroups blocks. Every group has one block of each row, so a pass over all of
// them is even; and at a place that moves from row to row by the golden ratio of a row, so that blocks some
// regular distance apart (a remainder in every 256th query: 0.2 ms on one compute unit for each 1024 of 640 slots,
// as group = block mod 256) do not all meet in one group.
RK_BOTH constexpr long long marked_block(unsigned row, unsigned group) {
    return (long long)row * kGaTargetGroups + ((group - (row * 0x9e3779b1u >> 24)) & (kGaTargetGroups - 1));
}

}  // namespace rk
