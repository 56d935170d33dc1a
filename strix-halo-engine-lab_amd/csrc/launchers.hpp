// Launches whose kernels live in translation units of their own (they compile in parallel).
#pragma once
#include "a8_rows.hpp"
#include "plan_block.hpp"
#include "prefill_args.hpp"
#include "q4k_rows.hpp"
#include "route_wave.hpp"

namespace strix950 {

// route.hip: logits of a batch past the decode sizes into a.scores; softmax, selection and weights of every row of a.scores
void launch_route_batch_logits(const RouteArgs& a, hipStream_t st);
void launch_route_select(const RouteArgs& a, hipStream_t st);
// RMSNorm of rows of any input kind into dense fp32 rows (weight may be null: a unit scale)
void launch_norm_rows(const void* x, uint32_t kind, uint64_t x_stride, const float* weight, uint32_t hidden, float eps, float* normed, uint32_t rows, hipStream_t st);
// A8 image, check of the routes and status words of the rows of a staged batch; q.status is not used.
struct RouteCheck {
    const uint32_t* routes; const float* route_weights;      // [rows][top_k]; weights may be null
    uint32_t experts, top_k;
    uint32_t *status, *job_status;
};
// plan (unless it has no experts): the expert plan of the rows' routes as well.
void launch_prologue_rows(const A8RowArgs& q, uint32_t kind, uint32_t rows, const RouteCheck& c, const PlanArgs& plan, hipStream_t st);

// prefill.hip: the most rows of a plan item for the products of a batch
uint32_t prefill_split(const mi355_moe_weights& wv, uint32_t assignments);
// prefill.hip: sub-block sums of the input rows, gate / up + SwiGLU and down rows of a planned batch. `a` holds everything but the
// products' own fields (weights, strides, k, features, tiles, units). check: the routes' check and the status words as well. plan: the batch's plan too.
void launch_prefill_products(const mi355_moe_weights& wv, PrefillArgs a, uint32_t rows, uint8_t* x_sums, const RouteCheck* check, const PlanArgs& plan,
                             uint32_t items_at, uint32_t order_at, hipStream_t st);

// q4k_mma.hip: experts on the int8 matrix cores (gate / up Q4_K or Q5_K; down Q4_K, Q6_K, or Q8_0 and Q5_1 rows of whole stages of 256 weights;
// dense batches Q4_K). dense: the rows of a one-expert batch (0: planned items); width: the most rows an
// item (or the dense batch) holds. The last leaves the raw gate and up values of a dense batch of at most 16 rows.
void launch_mma_project(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, uint32_t width, hipStream_t st);
void launch_mma_down(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, uint32_t width, hipStream_t st);
void launch_mma_gate_up_rows(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, hipStream_t st);

}  // namespace strix950
