// The matrix-core prefill of the routed experts: kernels of prefill_f16.hpp and prefill_reg.hpp, and the choice between them.
#include "host_common.hpp"
#include "launchers.hpp"
#include "prefill_reg.hpp"

namespace strix950 {

void launch_prefill_products(const mi355_moe_weights& wv, PrefillArgs a, uint32_t rows, uint8_t* x_sums, uint32_t items_at, uint32_t order_at, hipStream_t st) {
    token_sums_kernel<<<rows, 256, 0, st>>>(a.x, a.x_stride, wv.hidden, x_sums);
    if (pf_sum_slots(wv.ffn) != wv.ffn / 32U) clear_sum_padding_kernel<<<a.assignments, 64, 0, st>>>(a.h_sums, wv.ffn);
    const uint32_t item_slots = (a.items + 7U) / 8U * 8U;
    // persistent workgroups, as many as are resident: one per compute unit (LDS allows no second one) or `each` of the narrow form
    const uint32_t cus = compute_units();
    const uint32_t resident = (cus > 8U ? cus : 256U) & ~7U;
    const auto grid_of = [&](uint32_t units, uint32_t each = 1U) { return units < each * resident ? units : each * resident; };
    // Up to kNarrowRows rows per expert on average the narrow form of prefill_reg.hpp: two workgroups of half the width share a compute
    // unit, so one's start and end hide behind the other's products. Measured (wide, narrow): hidden 2048, ffn 768, 128 experts top-8, 64
    // rows 124, 108 us; 150 rows 160, 146 us; 333 rows 198, 191 us; 1200 rows 315, 362 us; hidden 4096, ffn 1536, 64 experts, 64 rows 272,
    // 246 us; 150 rows 312, 312 us; 333 rows 412, 438 us.
    constexpr uint64_t kNarrowRows = 24;
    const bool narrow = a.assignments <= kNarrowRows * wv.experts;
    // gate / up + SwiGLU. Q4_K tensors: every wave expands its own rows in registers (prefill_reg.hpp); Q5_K / Q8_0: the loader /
    // multiplier kernel (prefill_f16.hpp). Both leave h as two fp16 planes and its sub-block sums.
    a.wa = wv.gate; a.wb = wv.up; a.expert_stride = wv.gate_expert_stride; a.row_stride = wv.gate_row_stride; a.k = wv.hidden; a.features = wv.ffn;
    a.lo_pass = 0;
    if (wv.gate_type == MI355_TYPE_Q4_K && wv.ffn % 128U == 0) {
        a.tiles = wv.ffn / (narrow ? 64U : 128U); a.units = item_slots * a.tiles;
        if (narrow) prefill_reg_kernel<0, 4, 64><<<grid_of(2U * a.units, 2U), 256, 0, st>>>(a, items_at, order_at);
        else prefill_reg_kernel<0, 8, 128><<<grid_of(a.units), 512, 0, st>>>(a, items_at, order_at);
    } else {
        a.tiles = wv.ffn / 64U; a.units = item_slots * a.tiles;
        if (wv.gate_type == MI355_TYPE_Q8_0) prefill_f16_kernel<0, 1><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
        else if (wv.gate_type == MI355_TYPE_Q5_K) prefill_f16_kernel<0, 2><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
        else prefill_f16_kernel<0, 0><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
    }
    // down rows: h enters as hi + lo. The register-operand kernel multiplies both planes in one sweep of the weights; the loader /
    // multiplier kernel runs a second pass over the lo plane that adds to the first pass's outputs.
    a.wa = wv.down; a.wb = nullptr; a.expert_stride = wv.down_expert_stride; a.row_stride = wv.down_row_stride; a.k = wv.ffn; a.features = wv.hidden;
    if (wv.down_type == MI355_TYPE_Q4_K && wv.hidden % 256U == 0) {
        a.tiles = wv.hidden / (narrow ? 128U : 256U); a.units = item_slots * a.tiles;
        if (narrow) prefill_reg_kernel<1, 4, 64><<<grid_of(2U * a.units, 2U), 256, 0, st>>>(a, items_at, order_at);
        else prefill_reg_kernel<1, 8, 128><<<grid_of(a.units), 512, 0, st>>>(a, items_at, order_at);
    } else {
        a.tiles = wv.hidden / 128U; a.units = item_slots * a.tiles;
        for (uint32_t pass = 0; pass < 2U; ++pass) {
            a.lo_pass = pass;
            if (wv.down_type == MI355_TYPE_Q8_0) prefill_f16_kernel<1, 1><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
            else if (wv.down_type == MI355_TYPE_Q5_K) prefill_f16_kernel<1, 2><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
            else prefill_f16_kernel<1, 0><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
        }
    }
}

}  // namespace strix950
