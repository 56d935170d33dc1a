// The words of an expert plan (the workspace behind mi355_moe_rows.plan).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace strix950 {

// Plan words (uint32): [0] assignments A = rows * top_k, [1] touched experts U, [2] largest group, [3] launch ticket,
// [4] work items; [16, 272) ticket / scratch words; offsets[experts + 1]; touched[experts] (ids of the experts with work,
// ascending); order[A]: assignment indices (row * top_k + slot) grouped by expert, ascending row then slot inside an
// expert; items[A] x 4 words {expert, begin, end, 0}: the work items of the expert kernels, a touched expert's assignments
// cut into pieces of at most `split` (zero records after the last item, up to the launch's item bound).
// Reference: src/hip_moe_q4k_a8_probe.hip:91-147 (stable CSR of (row, slot) by expert).
__host__ __device__ constexpr uint32_t pad4(uint32_t v) { return (v + 3U) & ~3U; }
// ticket / scratch words right after the header, at the same place for every batch size (every launch leaves them zero, and a
// workspace is reused with varying row counts): [0, 16) row tickets of the fused router, [16, 32) its quantiser tickets,
// [128, 144) per-row A8 flags of the fused prologue
constexpr uint32_t kPlanTicketsAt = 16, kPlanTicketWords = 256;
// Behind the ticket words, also at a fixed place, the words of a decode batch planned from early routes (route_early.hpp):
//   one word per assignment (finished projection waves in the low half, bit 31 = non-finite projection);
//   one 64-bit tag per assignment {epoch, early expert};
//   three 128-byte lines per row (the 64-bit word {epoch, slots} that the row's side block leaves for its helpers, arrival counts of the A8
//     prologue blocks - with the row's flag word beside it - and of the exact router's side blocks) and a line with one tag per row (epoch of the call whose A8 image of that row is
//     complete) and the epoch word.
// Counts are zero when the plan is allocated and every launch leaves them zero. The epoch of a call is the epoch word + 1; the
// call's down launch stores it back, so tags of earlier calls never look current and nothing has to be reset.
constexpr uint32_t kLineWords = 32, kEarlyMaxAssignments = 128, kEarlyMinAssignments = 8, kEarlyMaxRows = 16;
constexpr uint32_t kPlanAwordsAt = kPlanTicketsAt + kPlanTicketWords, kPlanEtagsAt = kPlanAwordsAt + kEarlyMaxAssignments;
constexpr uint32_t kPlanLinesAt = (kPlanEtagsAt + 2U * kEarlyMaxAssignments + kLineWords - 1U) / kLineWords * kLineWords;      // (lines of a 128-byte aligned plan)
constexpr uint32_t kLinesVerdict = 0, kLinesPrologue = kEarlyMaxRows * kLineWords, kLinesSide = 2U * kEarlyMaxRows * kLineWords;
constexpr uint32_t kLinesRowTags = 3U * kEarlyMaxRows * kLineWords, kLinesEpoch = kLinesRowTags + kEarlyMaxRows;
constexpr uint32_t kPlanOffsetsAt = kPlanLinesAt + kLinesRowTags + kLineWords;
static_assert(kPlanEtagsAt % 2U == 0 && kPlanOffsetsAt % 4U == 0, "tags on 8 bytes, the plan arrays on 16");
__host__ __device__ constexpr uint32_t plan_touched_at(uint32_t experts) { return kPlanOffsetsAt + pad4(experts + 1U); }
__host__ __device__ constexpr uint32_t plan_order_at(uint32_t experts) { return plan_touched_at(experts) + pad4(experts); }
// most work items a plan can hold (layout) and most a launch with pieces of `split` assignments can produce (grid size)
__host__ __device__ constexpr uint32_t plan_item_capacity(uint32_t assignments) { return assignments; }
__host__ __device__ inline uint32_t plan_item_bound(uint32_t experts, uint32_t assignments, uint32_t split) {
    const uint32_t most = experts + assignments / split;
    return assignments < most ? assignments : most;
}
__host__ __device__ constexpr uint32_t plan_items_at(uint32_t experts, uint32_t assignments) { return plan_order_at(experts) + pad4(assignments); }
__host__ __device__ constexpr uint32_t plan_words_total(uint32_t experts, uint32_t assignments) {
    return plan_items_at(experts, assignments) + 4U * plan_item_capacity(assignments);
}

}  // namespace strix950
