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

// The start of a staged batch in one launch: the expert plan (a workgroup per expert), and a workgroup per row for the A8 image of the row, the
// check of its routes (by a wave of their own) and its status word. Bound by latency (a launch of this size costs about 4.5 us whatever it does).
template <int KIND>
__global__ __launch_bounds__(1024) void prologue_rows_kernel(A8RowArgs q, RouteCheck c, uint32_t image_threads, PlanArgs plan) {
    __shared__ PlanLds lds;
    if (blockIdx.x < plan.experts) return plan_block(lds, plan, blockIdx.x);
    if (threadIdx.x >= image_threads + 64U) return;
    const uint32_t row = blockIdx.x - plan.experts, lane = threadIdx.x & 63U;
    int bad_value = 0, bad_route = 0;
    if (threadIdx.x < image_threads) bad_value = a8_row<KIND>(q, row, image_threads);
    else {
        for (uint32_t k = lane; k < c.top_k; k += 64U) {
            if (c.routes[static_cast<size_t>(row) * c.top_k + k] >= c.experts) bad_route = 1;
            if (c.route_weights && !finite_f(c.route_weights[static_cast<size_t>(row) * c.top_k + k])) bad_route = 1;
        }
    }
    const uint32_t bits = (__syncthreads_or(bad_value) ? static_cast<uint32_t>(MI355_STATUS_NONFINITE_ACTIVATION) : 0U) |
                          (__syncthreads_or(bad_route) ? static_cast<uint32_t>(MI355_STATUS_INVALID_ROUTE) : 0U);
    if (threadIdx.x == 0) {
        c.status[row] = bits;
        if (row == 0) *c.job_status = 0;
    }
}

void launch_prologue_rows(const A8RowArgs& q, uint32_t kind, uint32_t rows, const RouteCheck& c, const PlanArgs& plan, hipStream_t st) {
    const uint32_t image = a8_row_threads(q.width) + 64U, used = image < 1024U ? image : 1024U;
    const uint32_t threads = plan.experts && used < 512U ? 512U : used, grid = plan.experts + rows;
    if (kind == MI355_INPUT_F32) prologue_rows_kernel<0><<<grid, threads, 0, st>>>(q, c, used - 64U, plan);
    else if (kind == MI355_INPUT_F16) prologue_rows_kernel<1><<<grid, threads, 0, st>>>(q, c, used - 64U, plan);
    else prologue_rows_kernel<2><<<grid, threads, 0, st>>>(q, c, used - 64U, plan);
}

void launch_route_select(const RouteArgs& a, hipStream_t st) { route_select_kernel<<<a.rows, 64, 0, st>>>(a); }

// RMSNorm of rows of any input kind into fp32 rows (in front of a layer that does not norm its rows in the router's launch), bit for bit rmsnorm_f32_kernel: lane l of L = 256
// (n >= 512) or 128 chains fma(x, x, a) over x[l], x[l + L], ...; the L partial sums are halved, l with l + 128, l + 64, ..., l + 1.
// A thread per chain. Bound by latency: the HELD first values of a chain and their weights are asked for at once and kept (one by one past
// the first eight, 1 row of 2048 fp16 values, 8 of 3072, 1 of 4096, 3 of 6144: 5.5, 8.5, 11, 16 us, now 2.2, 2.7, 4.7, 4.0), and every wave
// halves the sums by itself, in registers (1 barrier for 9).
template <int KIND, uint32_t HELD>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const uint8_t* x, uint64_t x_stride, const float* w, uint32_t n, float eps, float* y) {
    __shared__ float partial[256];
    const uint8_t* xr = x + blockIdx.x * x_stride;
    const uint32_t l = threadIdx.x, lane = l & 63U, L = n >= 512U ? 256U : 128U, end = l < L ? n : 0U;
    float v[HELD], wv[HELD], a = 0.0F;
#pragma unroll
    for (uint32_t j = 0; j < HELD; ++j) {
        const uint32_t i = min(l + L * j, n - 1U);  // (no branch a value: the conversion in it would wait for its load)
        v[j] = load_activation<KIND>(xr, i);
        wv[j] = w ? w[i] : 0.0F;
    }
#pragma unroll
    for (uint32_t j = 0; j < HELD; ++j)
        if (l + L * j < end) a = __builtin_fmaf(v[j], v[j], a);
    for (uint32_t i = l + L * HELD; i < end; i += L) {
        const float u = load_activation<KIND>(xr, i);
        a = __builtin_fmaf(u, u, a);
    }
    partial[l] = a;
    __syncthreads();
    float sum = L == 256U ? (partial[lane] + partial[lane + 128U]) + (partial[lane + 64U] + partial[lane + 192U]) : partial[lane] + partial[lane + 64U];
    sum = sum + __shfl_xor(sum, 32);
    sum = sum + xor16_f(sum); sum = sum + xor8_f(sum); sum = sum + xor4_f(sum); sum = sum + xor2_f(sum); sum = sum + xor1_f(sum);
    const float r = 1.0F / __builtin_sqrtf(sum / static_cast<float>(n) + eps);
    float* yr = y + static_cast<size_t>(blockIdx.x) * n;
#pragma unroll
    for (uint32_t j = 0; j < HELD; ++j)
        if (l + L * j < end) { const float u = v[j] * r; yr[l + L * j] = w ? u * wv[j] : u; }
    for (uint32_t i = l + L * HELD; i < end; i += L) {
        const float u = load_activation<KIND>(xr, i) * r;
        yr[i] = w ? u * w[i] : u;
    }
}

void launch_norm_rows(const void* x, uint32_t kind, uint64_t x_stride, const float* weight, uint32_t hidden, float eps, float* normed, uint32_t rows, hipStream_t st) {
    const uint8_t* at = static_cast<const uint8_t*>(x);
    const auto launch = [&](auto held) {
        constexpr uint32_t HELD = decltype(held)::value;
        if (kind == MI355_INPUT_F32) rmsnorm_rows_kernel<0, HELD><<<rows, 256, 0, st>>>(at, x_stride, weight, hidden, eps, normed);
        else if (kind == MI355_INPUT_F16) rmsnorm_rows_kernel<1, HELD><<<rows, 256, 0, st>>>(at, x_stride, weight, hidden, eps, normed);
        else rmsnorm_rows_kernel<2, HELD><<<rows, 256, 0, st>>>(at, x_stride, weight, hidden, eps, normed);
    };
    if (hidden <= 2048U) launch(std::integral_constant<uint32_t, 8>{});
    else if (hidden <= 4096U) launch(std::integral_constant<uint32_t, 16>{});
    else launch(std::integral_constant<uint32_t, 32>{});
}

}  // namespace strix950
