// The matrix-core prefill of the routed experts: kernels of prefill_f16.hpp and prefill_reg.hpp, and the choice between them.
#include "host_common.hpp"
#include "launchers.hpp"
#include "prefill_reg.hpp"

namespace strix950 {

// What a batch needs besides its plan before the products, one workgroup per row: the row's sub-block sums (a thread per sub-block of 32,
// fp32 sum in index order), zeros in the padding slots of the sums of h of the row's assignments (ffn / 32 not a multiple of 16; every
// assignment has a row of sums, whichever order the plan gives them), and - with a check - the routes' check and the status words.
// Bound by latency: one launch in the place of three (333 rows: about 4.5 us each).
__global__ __launch_bounds__(256) void prefill_prologue_kernel(const uint8_t* x, uint64_t x_stride, uint32_t k, uint8_t* x_sums, uint8_t* h_sums, uint32_t ffn,
                                                               uint32_t top_k, RouteCheck check) {
    const uint32_t row = blockIdx.x, slots = pf_sum_slots(k), h_slots = pf_sum_slots(ffn), h_used = ffn / 32U, pad = h_slots - h_used;
    _Float16* hi = reinterpret_cast<_Float16*>(x_sums + static_cast<size_t>(row) * pf_sum_row_bytes(k));
    _Float16* lo = hi + slots;
    for (uint32_t s = threadIdx.x; s < slots; s += 256U) {
        float sum = 0.0F;
        if (s < k / 32U) {
            const half8* p = reinterpret_cast<const half8*>(x + static_cast<size_t>(row) * x_stride + 64U * s);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const half8 v = p[i];
#pragma unroll
                for (int j = 0; j < 8; ++j) sum += static_cast<float>(v[j]);
            }
        }
        split_half(sum, hi[s], lo[s]);
    }
    for (uint32_t i = threadIdx.x; i < pad * top_k; i += 256U) {
        const uint32_t slot = i / pad, s = h_used + i - slot * pad;
        _Float16* out = reinterpret_cast<_Float16*>(h_sums + (static_cast<size_t>(row) * top_k + slot) * pf_sum_row_bytes(ffn));
        out[s] = static_cast<_Float16>(0.0F);
        out[h_slots + s] = static_cast<_Float16>(0.0F);
    }
    if (!check.status || threadIdx.x < 192U) return;
    uint32_t bad = 0;
    for (uint32_t i = threadIdx.x - 192U; i < top_k; i += 64U) {
        if (check.routes[static_cast<size_t>(row) * top_k + i] >= check.experts) bad = 1;
        if (check.route_weights && !finite_f(check.route_weights[static_cast<size_t>(row) * top_k + i])) bad = 1;
    }
    const bool any = __ballot(bad) != 0;
    if (threadIdx.x == 192U) {
        check.status[row] = any ? static_cast<uint32_t>(MI355_STATUS_INVALID_ROUTE) : 0U;
        if (row == 0) *check.job_status = 0;
    }
}

namespace {
// Which Q4_K batches the four-wave form of prefill_reg.hpp serves. It sweeps an expert's weights once per 32 rows, the wide form once per
// 128; it has three times the workgroups in flight. Measured (wide, four waves), rows per expert on average and rounds of the wide form's
// gate / up workgroups beside them: 8.5, 5.8 256, 199 us; 12.3, 13 185, 168; 15, 8.4 776, 707; 21, 3.5 195, 178; 22, 14 965, 1028;
// 25, 9 867, 894; 37, 7.8 879, 961; 40, 3.3 435, 419; 46, 1.8 414, 380; 50, 4.2 270, 275; 56, 4.0 194, 178; 45, 18 1847, 2312.
bool few_rows(const mi355_moe_weights& wv, uint32_t assignments) {
    const uint64_t e = wv.experts, a = assignments;
    return a <= 16ULL * e || (a <= 56ULL * e && (128ULL * e + a) * wv.ffn <= 4ULL * compute_units() * 128U * 128U);
}
bool reg_gate(const mi355_moe_weights& wv) { return wv.gate_type == MI355_TYPE_Q4_K && wv.ffn % 128U == 0; }
bool reg_down(const mi355_moe_weights& wv) { return wv.down_type == MI355_TYPE_Q4_K && wv.hidden % 256U == 0; }
}  // namespace

uint32_t prefill_split(const mi355_moe_weights& wv, uint32_t assignments) {
    return reg_gate(wv) && reg_down(wv) && few_rows(wv, assignments) ? 32U : kPfTile;
}

void launch_prefill_products(const mi355_moe_weights& wv, PrefillArgs a, uint32_t rows, uint8_t* x_sums, const RouteCheck* check, uint32_t items_at, uint32_t order_at, hipStream_t st) {
    prefill_prologue_kernel<<<rows, 256, 0, st>>>(a.x, a.x_stride, wv.hidden, x_sums, a.h_sums, wv.ffn, wv.top_k, check ? *check : RouteCheck{});
    const uint32_t item_slots = (a.items + 7U) / 8U * 8U;
    // persistent workgroups, as many as are resident: one per compute unit (LDS allows no second one) or `each` of the four-wave form
    const uint32_t cus = compute_units();
    const uint32_t resident = (cus > 8U ? cus : 256U) & ~7U;
    const auto grid_of = [&](uint32_t units, uint32_t each = 1U) { return units < each * resident ? units : each * resident; };
    const bool few = few_rows(wv, a.assignments);
    a.subs = prefill_split(wv, a.assignments) / 32U;
    // gate / up + SwiGLU. Q4_K tensors: every wave expands its own rows in registers (prefill_reg.hpp); Q5_K / Q8_0: the loader /
    // multiplier kernel (prefill_f16.hpp). Both leave h as two fp16 planes and its sub-block sums.
    a.wa = wv.gate; a.wb = wv.up; a.expert_stride = wv.gate_expert_stride; a.row_stride = wv.gate_row_stride; a.k = wv.hidden; a.features = wv.ffn;
    a.lo_pass = 0;
    if (reg_gate(wv)) {
        a.tiles = wv.ffn / (few ? 64U : 128U); a.units = item_slots * a.tiles;
        if (few) prefill_reg_kernel<0, 4><<<grid_of(a.subs * a.units, 3U), 256, 0, st>>>(a, items_at, order_at);
        else prefill_reg_kernel<0, 8><<<grid_of(a.units), 512, 0, st>>>(a, items_at, order_at);
    } else {
        a.tiles = wv.ffn / 64U; a.units = item_slots * a.tiles;
        if (wv.gate_type == MI355_TYPE_Q8_0) prefill_f16_kernel<0, 1><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
        else if (wv.gate_type == MI355_TYPE_Q5_K) prefill_f16_kernel<0, 2><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
        else prefill_f16_kernel<0, 0><<<grid_of(a.units), kPfThreads, 0, st>>>(a, items_at, order_at);
    }
    // down rows: h enters as hi + lo. The register-operand kernel multiplies both planes in one sweep of the weights; the loader /
    // multiplier kernel runs a second pass over the lo plane that adds to the first pass's outputs.
    a.wa = wv.down; a.wb = nullptr; a.expert_stride = wv.down_expert_stride; a.row_stride = wv.down_row_stride; a.k = wv.ffn; a.features = wv.hidden;
    if (reg_down(wv)) {
        a.tiles = wv.hidden / (few ? 128U : 256U); a.units = item_slots * a.tiles;
        if (few) prefill_reg_kernel<1, 4><<<grid_of(a.subs * a.units, 3U), 256, 0, st>>>(a, items_at, order_at);
        else prefill_reg_kernel<1, 8><<<grid_of(a.units), 512, 0, st>>>(a, items_at, order_at);
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
