// The matrix-core prefill of the routed experts: the kernels of prefill_reg.hpp and the choice between their forms.
#include "host_common.hpp"
#include "launchers.hpp"
#include "prefill_reg.hpp"

#include <atomic>

namespace strix950 {

// What a batch needs before the products: the expert plan (a workgroup per expert), and a workgroup per row for the row's sub-block sums (a thread per
// sub-block of 32, fp32 sum in index order) and - with a check - the routes' check and the status words.
// Bound by latency: one launch in the place of three (333 rows: about 4.5 us each).
__global__ __launch_bounds__(512) void prefill_prologue_kernel(const uint8_t* x, uint64_t x_stride, uint32_t k, uint8_t* x_sums, uint32_t top_k, RouteCheck check, PlanArgs plan) {
    __shared__ PlanLds lds;
    if (blockIdx.x < plan.experts) return plan_block(lds, plan, blockIdx.x);
    if (threadIdx.x >= 256U) return;
    const uint32_t row = blockIdx.x - plan.experts;
    _Float16* hi = reinterpret_cast<_Float16*>(x_sums + static_cast<size_t>(row) * pf_sum_row_bytes(k));
    _Float16* lo = hi + pf_sum_slots(k);
    for (uint32_t s = threadIdx.x; s < k / 32U; s += 256U) {
        float sum = 0.0F;
        const half8* p = reinterpret_cast<const half8*>(x + static_cast<size_t>(row) * x_stride + 64U * s);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const half8 v = p[i];
#pragma unroll
            for (int j = 0; j < 8; ++j) sum += static_cast<float>(v[j]);
        }
        split_half(sum, hi[s], lo[s]);
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
// Which batches the four-wave form of prefill_reg.hpp serves. It sweeps an expert's weights once per 32 rows, the wide form once per
// 128; it has three times the workgroups in flight. Measured (wide, four waves), rows per expert on average and rounds of the wide form's
// gate / up workgroups beside them: 8.5, 5.8 256, 199 us; 12.3, 13 185, 168; 15, 8.4 776, 707; 21, 3.5 195, 178; 22, 14 965, 1028;
// 25, 9 867, 894; 37, 7.8 879, 961; 40, 3.3 435, 419; 46, 1.8 414, 380; 50, 4.2 270, 275; 56, 4.0 194, 178; 45, 18 1847, 2312.
// Q8_0 rows are twice as wide, and the down rows are swept twice: up to 13 rows per expert, while rows times rounds are few, or the rows of an
// expert, or the rows short, so that a workgroup's start is what it waits for. Measured the same way, hidden 2048 and more:
// 4, 3.1 175, 148; 9.4, 3.2 467, 451; 9.4, 3.2 236, 225; 13, 3.3 247, 239; 6, 4.2 523, 449; 9.4, 4.3 536, 520; 13, 4.4 567, 645; 5, 5.2 316, 285;
// 9, 5.4 340, 348; 12, 5.4 578, 656; 7, 6.3 363, 351; 9, 6.4 384, 397; 3.8, 7.7 910, 886; 6, 7.9 1055, 1107; 12.5, 8.2 1238, 1348; 2, 16 479, 420;
// 4, 17 535, 509; 6, 17 566, 596; 9, 17 579, 694; hidden 1280, 13, 4.1 166, 128; hidden 1024, 13, 6.2 179, 148. Past 13 rows per expert: 21, 3.5 257, 285; 25, 3.6
// 538, 615; 37, 3.9 325, 369; in one round 25, 0.9 123, 95; 37, 1.0 128, 120; 50, 0.7 134, 119.
// Measured again for 50 to 80 rows per expert (rows, rounds, wide, four waves): Q4_K 62, 1.1 152, 129; 70, 1.5 142, 127; 70, 0.5 198, 162; 75, 1.6 258, 226; 77, 2.0 301, 260;
// 78, 1.5 124, 134; 94, 2.6 205, 213; 150, 2.2 309, 355; Q5_K 62, 1.1 170, 159; 70, 1.5 156, 152; 75, 1.6 299, 294; Q8_0 62, 0.7 114, 95; 70, 0.5 268, 245; 75, 0.9 192, 213;
// 75, 1.0 150, 166.
// However many rows an expert has, while the four-wave form's units (of 32 rows) find room at once, three workgroups a compute unit, which the wide
// form's leave mostly idle. Units, then the same two times, one expert: Q4_K hidden 2048 / ffn 768, 56 86.5, 50.9; 154 86.6, 52.4; 448 91.3, 67.0; 4096 /
// 2048, 224 146, 79.9; Q8_0 56 109, 55.7; 448 116, 84.6; 224 201, 98.4; Q5_K 448 99.9, 74.7; 224 168, 93.4; of 16 and 32 experts Q4_K 728 95.3, 81.3; 728 70.7, 57.3;
// Q5_K 728 102, 92.0; Q8_0 728 84.8, 72.4. Past that: Q4_K 928 73.4, 64.9; 1024 156, 155; 1106 112, 109; 1344 106, 110; Q8_0 928 86.2, 85.8; 1024 212, 257; 1106 133,
// 147; Q5_K 1024 177, 196; 1106 119, 122.
bool few_rows(const mi355_moe_weights& wv, uint32_t assignments) {
    const uint64_t items = (assignments + 16ULL * wv.experts + 31ULL) / 32U, tiles = wv.ffn / 64U + wv.hidden / 128U;          // (of both launches: twice the units)
    if (items * tiles <= 6ULL * compute_units()) return true;
    const uint64_t e = wv.experts, a = assignments, work = (128ULL * e + a) * wv.ffn, round = compute_units() * 128ULL * 128U;
    if (wv.gate_type == MI355_TYPE_Q8_0 || wv.down_type == MI355_TYPE_Q8_0) {
        const bool starts = a * work <= 51ULL * e * round || 2ULL * a <= 9ULL * e || wv.hidden <= 1280U;
        return (a <= 13ULL * e && starts) || (a <= 70ULL * e && work <= round);
    }
    return a <= 16ULL * e || (a <= 56ULL * e && work <= 4ULL * round) || (a <= 75ULL * e && work <= 2ULL * round);
}
}  // namespace

std::atomic<uint32_t> g_prefill_form{0};

uint32_t prefill_split(const mi355_moe_weights& wv, uint32_t assignments) {
    const uint32_t form = g_prefill_form.load(std::memory_order_relaxed);
    return (form ? form == 1U : few_rows(wv, assignments)) ? kPfFewRows : kPfTile;
}

void launch_prefill_products(const mi355_moe_weights& wv, PrefillArgs a, uint32_t rows, uint8_t* x_sums, const RouteCheck* check, const PlanArgs& plan, uint32_t items_at, uint32_t order_at, hipStream_t st) {
    prefill_prologue_kernel<<<plan.experts + rows, 512, 0, st>>>(a.x, a.x_stride, wv.hidden, x_sums, wv.top_k, check ? *check : RouteCheck{}, plan);
    const uint32_t item_slots = (a.items + 7U) / 8U * 8U;
    // persistent workgroups, as many as are resident: one per compute unit (LDS allows no second one) or `each` of the four-wave form
    const uint32_t cus = compute_units();
    const uint32_t resident = (cus > 8U ? cus : 256U) & ~7U;
    const auto grid_of = [&](uint32_t units, uint32_t each = 1U) { return units < each * resident ? units : each * resident; };
    const bool few = plan.split == kPfFewRows;          // (the form that the plan's items are made for)
    const auto launch = [&](auto mode, uint32_t type) {
        constexpr int M = decltype(mode)::value;
        const auto of = [&](auto format) {
            constexpr int F = decltype(format)::value;
            if (few) prefill_reg_kernel<M, 4, F><<<grid_of(a.units, 3U), 256, 0, st>>>(a, items_at, order_at);
            else prefill_reg_kernel<M, 8, F><<<grid_of(a.units), 512, 0, st>>>(a, items_at, order_at);
        };
        if (type == MI355_TYPE_Q8_0) of(std::integral_constant<int, kRgQ80>{});
        else if (type == MI355_TYPE_Q5_K) of(std::integral_constant<int, kRgQ5K>{});
        else of(std::integral_constant<int, kRgQ4K>{});
    };
    // gate / up + SwiGLU: leaves h as two fp16 planes and its sub-block sums
    a.wa = wv.gate; a.wb = wv.up; a.expert_stride = wv.gate_expert_stride; a.row_stride = wv.gate_row_stride; a.k = wv.hidden; a.features = wv.ffn;
    a.tiles = wv.ffn / (few ? 64U : 128U); a.units = item_slots * a.tiles;
    launch(std::integral_constant<int, 0>{}, wv.gate_type);
    // down rows: h enters as hi + lo, both planes in one sweep of the weights (Q4_K) or in two of one launch
    a.wa = wv.down; a.wb = nullptr; a.expert_stride = wv.down_expert_stride; a.row_stride = wv.down_row_stride; a.k = wv.ffn; a.features = wv.hidden;
    a.tiles = wv.hidden / (few ? 128U : 256U); a.units = item_slots * a.tiles;
    launch(std::integral_constant<int, 1>{}, wv.down_type);
}

}  // namespace strix950

extern "C" void mi355_debug_prefill_form(uint32_t form) { strix950::g_prefill_form.store(form, std::memory_order_relaxed); }
