// Q4_K experts on the int8 matrix cores (q4k_mma_moe.hpp): which instance serves a launch.
#include "host_common.hpp"
#include "launchers.hpp"
#include "q4k_mma_moe.hpp"

namespace strix950 {

template <int NAL>
inline void launch_mma_project_nal(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, hipStream_t st) {
    const dim3 grid(w.ffn / 32U, dense ? (dense + 2U * NAL - 1U) / (2U * NAL) : items);
    q4k_mma_project_kernel<NAL, (NAL >= 8 ? 2 : 3)><<<grid, 256, 0, st>>>(w, r, rows * w.top_k, dense);
}
// A launch with no more workgroups than compute units (few, long rows) runs four stages of a tile at a time (measured at 5120
// rows x 27648, 8 rows: 59 -> 33 us; ring depths 2..4 within 2 us of each other in both forms).
template <int NAL>
inline void launch_mma_down_nal(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, hipStream_t st) {
    const dim3 grid(w.hidden / kMmaRows, dense ? (dense + 2U * NAL - 1U) / (2U * NAL) : items);
    if constexpr (NAL <= 8) {
        if (static_cast<uint64_t>(grid.x) * grid.y <= compute_units()) {
            q4k_mma_down_kernel<NAL, 2, 4><<<grid, 1024, 0, st>>>(w, r, rows * w.top_k, dense);
            return;
        }
    }
    q4k_mma_down_kernel<NAL, (NAL >= 8 ? 2 : 3), 1><<<grid, 256, 0, st>>>(w, r, rows * w.top_k, dense);
}
// width: the most rows an item (or the dense batch) holds
void launch_mma_project(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, uint32_t width, hipStream_t st) {
    if (width <= 4U) launch_mma_project_nal<2>(w, r, rows, dense, items, st);
    else if (width <= 8U) launch_mma_project_nal<4>(w, r, rows, dense, items, st);
    else if (width <= 16U) launch_mma_project_nal<8>(w, r, rows, dense, items, st);
    else launch_mma_project_nal<16>(w, r, rows, dense, items, st);
}
// (the down rows run best 16 rows to a sweep: 4096 rows over 256 experts, hidden 4096 / ffn 2048: 2.57 ms against 3.03 ms with 32)
void launch_mma_down(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, uint32_t width, hipStream_t st) {
    if (width <= 4U) launch_mma_down_nal<2>(w, r, rows, dense, items, st);
    else if (width <= 8U) launch_mma_down_nal<4>(w, r, rows, dense, items, st);
    else launch_mma_down_nal<8>(w, r, rows, dense, items, st);
}
void launch_mma_gate_up_rows(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, hipStream_t st) {
    const dim3 grid(w.ffn / kMmaRows, 1, 2);
    if (rows <= 8U) q4k_mma_down_kernel<4, 3, 1, true><<<grid, 256, 0, st>>>(w, r, rows, rows);
    else q4k_mma_down_kernel<8, 2, 1, true><<<grid, 256, 0, st>>>(w, r, rows, rows);
}

}  // namespace strix950
