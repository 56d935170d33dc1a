// The router of batches past the decode sizes: logits on the fp32 matrix cores (route_mma.hpp), softmax and selection per row.
#include "host_common.hpp"
#include "launchers.hpp"
#include "route_mma.hpp"


namespace strix950 {

// Logits in the 32-lane order: blocks of 8 experts x 8 rows.
template <int KIND>
__global__ __launch_bounds__(64) void route_logits_kernel(RouteArgs a) {
    __shared__ RouteLds lds;
    const uint32_t neb = (a.p.experts + 7U) / 8U;
    route_logits_block<KIND>(lds, a, (blockIdx.x % neb) * 8U, (blockIdx.x / neb) * 8U);
}

// softmax / top-k / weights, one row per one-wave block (the plain router).
__global__ __launch_bounds__(64) void route_select_kernel(RouteArgs a) {
    __shared__ __attribute__((aligned(16))) float sel_p[kRouteMaxExperts];
    route_select_row(sel_p, a, blockIdx.x);
}

void launch_route_batch_logits(const RouteArgs& a, hipStream_t st) {
    if (a.p.logits_order == MI355_LOGITS_FMA_ASCENDING && (a.rows + 15U) / 16U <= 65535U) return launch_route_mma(a, compute_units(), st);
    const uint32_t blocks = (a.p.experts + 7U) / 8U * ((a.rows + 7U) / 8U);
    if (a.kind == MI355_INPUT_F32) route_logits_kernel<0><<<blocks, 64, 0, st>>>(a);
    else if (a.kind == MI355_INPUT_F16) route_logits_kernel<1><<<blocks, 64, 0, st>>>(a);
    else route_logits_kernel<2><<<blocks, 64, 0, st>>>(a);
}

void launch_route_select(const RouteArgs& a, hipStream_t st) { route_select_kernel<<<a.rows, 64, 0, st>>>(a); }

}  // namespace strix950
