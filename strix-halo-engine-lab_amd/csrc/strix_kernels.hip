// MI355X (gfx950, wave64) kernels and C ABI of the quantized weight-product path. See include/mi355_strix.h for the
// contract of every entry point; reference file:line citations are relative to the reference tree.
#include "mi355_strix.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "device_math.hpp"
#include "host_common.hpp"
#include "launchers.hpp"
#include "plan_block.hpp"
#include "plan_layout.hpp"
#include "q4k_rows.hpp"
#include "q4k_blocks.hpp"
#include "q4k_pairs.hpp"
#include "q4k_quads.hpp"
#include "down_groups.hpp"
#include "q5k_quads.hpp"
#include "q6k_quads.hpp"
#include "route_wave.hpp"
#include "route_early.hpp"

namespace strix950 {

// ======================================================================================================== block decode
// One thread per output element. Q4_K: y = (d * sc) * q - (dmin * m), two products and one subtraction
// (src/ggml_dequant.cpp:119-130); Q8_0: y = int8 * d (src/ggml_dequant.cpp:84-87).
__device__ __forceinline__ void q4k_scale_min(const uint8_t* q, uint32_t j, uint32_t& sc, uint32_t& m) {
    if (j < 4) { sc = q[j] & 63U; m = q[j + 4] & 63U; }
    else { sc = (q[j + 4] & 0xFU) | ((q[j - 4] >> 6) << 4); m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4); }
}

__global__ __launch_bounds__(256) void dequantize_rows_kernel(uint32_t type, const uint8_t* rows, uint64_t row_stride,
                                                              uint32_t elements, float* out, uint64_t out_stride) {
    const uint32_t r = blockIdx.y;
    const uint8_t* row = rows + r * row_stride;
    for (uint32_t i = blockIdx.x * 256U + threadIdx.x; i < elements; i += gridDim.x * 256U) {
        float y;
        if (type == MI355_TYPE_Q8_0) {
            const uint8_t* b = row + (i / 32U) * kQ80Block;
            const float d = half_bits_to_float(b[0] | (static_cast<uint32_t>(b[1]) << 8));
            y = static_cast<float>(static_cast<int8_t>(b[2 + (i % 32U)])) * d;
        } else {
            const uint8_t* b = row + (i / 256U) * kQ4kBlock;
            const uint32_t k = i % 256U, j = k / 32U, l = k % 32U;
            uint32_t sc, m;
            q4k_scale_min(b + 4, j, sc, m);
            const float d = half_bits_to_float(b[0] | (static_cast<uint32_t>(b[1]) << 8));
            const float mn = half_bits_to_float(b[2] | (static_cast<uint32_t>(b[3]) << 8));
            const float d1 = d * static_cast<float>(sc), m1 = mn * static_cast<float>(m);
            const uint32_t byte = b[16 + 32 * (j / 2) + l];
            const float q = static_cast<float>((j & 1U) ? (byte >> 4) : (byte & 15U));
            y = d1 * q - m1;
        }
        out[r * out_stride + i] = y;
    }
}

// ======================================================================================================== weight writers
// Q8_0: include/strix/q8_0_rule.hpp:25-33 (d = amax / 127, id = 1 / d, q = roundf(v * id), d stored as fp16).
__global__ __launch_bounds__(256) void quantize_q8_0_rows_kernel(const float* x, uint64_t blocks, uint8_t* out) {
    for (uint64_t b = blockIdx.x * 256ULL + threadIdx.x; b < blocks; b += 256ULL * gridDim.x) {
        const float* v = x + b * 32;
        float amax = 0.0F;
        for (int j = 0; j < 32; ++j) amax = __builtin_fmaxf(amax, __builtin_fabsf(v[j]));
        const float d = amax / 127.0F;
        const float id = d != 0.0F ? 1.0F / d : 0.0F;
        uint8_t* o = out + b * kQ80Block;
        const uint32_t h = float_to_half_bits(d);
        o[0] = static_cast<uint8_t>(h); o[1] = static_cast<uint8_t>(h >> 8);
        for (int j = 0; j < 32; ++j) o[2 + j] = static_cast<uint8_t>(static_cast<int8_t>(static_cast<int>(__builtin_roundf(v[j] * id))));
    }
}

// Q4_K min/max writer (no reference counterpart; the reference only reads GGUF). Per 32-value sub-block: scale =
// (max - min) / 15 and offset = 0 - min with min clamped to <= 0; super-block d = max scale / 63, dmin = max offset / 63,
// both stored as fp16; 6-bit factors and 4-bit codes by round-to-nearest against the fp16-rounded d / dmin.
__global__ __launch_bounds__(64) void quantize_q4_k_rows_kernel(const float* x, uint64_t blocks, uint8_t* out) {
    for (uint64_t b = blockIdx.x * 64ULL + threadIdx.x; b < blocks; b += 64ULL * gridDim.x) {
        const float* v = x + b * 256;
        uint8_t* o = out + b * kQ4kBlock;
        float scale[8], offset[8], smax = 0.0F, omax = 0.0F;
        for (int j = 0; j < 8; ++j) {
            float lo = 0.0F, hi = v[32 * j];
            for (int l = 0; l < 32; ++l) { lo = __builtin_fminf(lo, v[32 * j + l]); hi = __builtin_fmaxf(hi, v[32 * j + l]); }
            hi = __builtin_fmaxf(hi, lo);
            scale[j] = (hi - lo) / 15.0F; offset[j] = 0.0F - lo;
            smax = __builtin_fmaxf(smax, scale[j]); omax = __builtin_fmaxf(omax, offset[j]);
        }
        const uint32_t dh = float_to_half_bits(smax / 63.0F), mh = float_to_half_bits(omax / 63.0F);
        const float d = half_bits_to_float(dh), dm = half_bits_to_float(mh);
        uint32_t sc[8], mn[8];
        for (int j = 0; j < 8; ++j) {
            sc[j] = d > 0.0F ? static_cast<uint32_t>(__builtin_fminf(63.0F, __builtin_rintf(scale[j] / d))) : 0U;
            mn[j] = dm > 0.0F ? static_cast<uint32_t>(__builtin_fminf(63.0F, __builtin_rintf(offset[j] / dm))) : 0U;
        }
        o[0] = static_cast<uint8_t>(dh); o[1] = static_cast<uint8_t>(dh >> 8);
        o[2] = static_cast<uint8_t>(mh); o[3] = static_cast<uint8_t>(mh >> 8);
        for (int j = 0; j < 4; ++j) {
            o[4 + j] = static_cast<uint8_t>((sc[j] & 63U) | ((sc[j + 4] >> 4) << 6));
            o[8 + j] = static_cast<uint8_t>((mn[j] & 63U) | ((mn[j + 4] >> 4) << 6));
            o[12 + j] = static_cast<uint8_t>((sc[j + 4] & 15U) | ((mn[j + 4] & 15U) << 4));
        }
        for (int p = 0; p < 4; ++p) {
            const float ed0 = d * static_cast<float>(sc[2 * p]), em0 = dm * static_cast<float>(mn[2 * p]);
            const float ed1 = d * static_cast<float>(sc[2 * p + 1]), em1 = dm * static_cast<float>(mn[2 * p + 1]);
            for (int l = 0; l < 32; ++l) {
                float r0 = 0.0F, r1 = 0.0F;
                if (ed0 > 0.0F) r0 = __builtin_fminf(15.0F, __builtin_fmaxf(0.0F, __builtin_rintf((v[64 * p + l] + em0) / ed0)));
                if (ed1 > 0.0F) r1 = __builtin_fminf(15.0F, __builtin_fmaxf(0.0F, __builtin_rintf((v[64 * p + 32 + l] + em1) / ed1)));
                o[16 + 32 * p + l] = static_cast<uint8_t>(static_cast<uint32_t>(r0) | (static_cast<uint32_t>(r1) << 4));
            }
        }
    }
}

// ======================================================================================================== A8 quantiser
// RMSNorm of fp32 rows in the reference's declared order (src/cpu/core/reference.cpp:86-103, lane count
// src/cpu/core/backend.hpp:91): lane l of L = 256 (n >= 512) or 128 runs the fma chain over x[l], x[l + L], ...; the L partial
// sums are halved in LDS (partial[l] += partial[l + h], h = L/2 .. 1); r = 1 / sqrt(sum / n + eps); y = (x * r) * w.
// One workgroup of L threads per row: the lanes' strided chains are coalesced reads as they stand.
__global__ __launch_bounds__(256) void rmsnorm_f32_kernel(const float* x, const float* w, uint32_t n, float eps, float* y) {
    __shared__ float partial[256];
    const uint32_t lanes = blockDim.x, lane = threadIdx.x;
    const float* xr = x + static_cast<size_t>(blockIdx.x) * n;
    float* yr = y + static_cast<size_t>(blockIdx.x) * n;
    float a = 0.0F;
    for (uint32_t i = lane; i < n; i += lanes) a = __builtin_fmaf(xr[i], xr[i], a);
    partial[lane] = a;
    for (uint32_t h = lanes / 2U; h > 0; h >>= 1) {
        __syncthreads();
        if (lane < h) partial[lane] = partial[lane] + partial[lane + h];
    }
    __syncthreads();
    const float r = 1.0F / __builtin_sqrtf(partial[0] / static_cast<float>(n) + eps);
    for (uint32_t i = lane; i < n; i += lanes) yr[i] = w ? (xr[i] * r) * w[i] : xr[i] * r;
}

// ======================================================================================================== router
// A8 prologue block qb of a fused decode launch (src/cpu/core/reference.cpp:35-55): two groups of 32 at a time, 8 groups per
// block; the last of a row's blocks publishes the row's status word.
// Row r counts its finished blocks in ticket[r * stride] and collects its flags in flags[r * stride]. LINES: the words are reached
// by device-scope atomics only and the count is a plain arrival (route_early.hpp); otherwise the count is an acquire-release ticket.
// NORM: the image of the row's RMSNorm, which is left in a.normed too (a block's eight groups are of one row: hidden % 256 == 0).
template <int KIND, bool NORM, bool LINES = false>
__device__ __forceinline__ void a8_prologue_block(const RouteArgs& a, uint32_t qb, uint32_t* ticket, uint32_t* flags, uint32_t stride,
                                                  uint32_t* row_tag = nullptr, uint32_t epoch = 0) {
    const uint32_t lane = threadIdx.x;
    {
        const uint32_t groups = a.hidden / 32U, total = a.rows * groups, g0 = qb * 8U;
        float factor = 1.0F;
        if constexpr (NORM) {
            float held[kNormHeld];
            norm_ask<KIND>(held, a.x + (g0 / groups) * a.x_stride, a.hidden);
            factor = norm_factor(held, a.hidden, a.norm_eps);
        }
        for (uint32_t i = 0; i < 8U; i += 2U) {
            const uint32_t g = g0 + i + (lane >> 5), j = lane & 31U;
            if (g < total) {
                const uint32_t r = g / groups, gi = g % groups;
                float v = load_activation<KIND>(a.x + r * a.x_stride, gi * 32U + j);
                if constexpr (NORM) {
                    v = v * factor;
                    if (a.norm_w) v = v * a.norm_w[gi * 32U + j];
                    a.normed[static_cast<size_t>(r) * a.hidden + gi * 32U + j] = v;
                }
                const float amax = max32(__builtin_fabsf(v));
                const bool tiny = amax > 0.0F && amax < 0x1p-119F;
                const float delta = (amax == 0.0F || tiny) ? 1.0F : amax / 127.0F;
                const int code = a8_code(v, delta, tiny);
                const int sum = sum32_i(code);
                const int bad = or32_i(finite_f(v) ? 0 : 1);
                store_shared_or_plain(LINES, a.codes + static_cast<size_t>(r) * a.hidden + gi * 32U + j, static_cast<int8_t>(code));
                if (j == 0) {
                    store_shared_or_plain(LINES, a.deltas + static_cast<size_t>(r) * groups + gi, delta);
                    store_shared_or_plain(LINES, a.sums + static_cast<size_t>(r) * groups + gi, static_cast<int32_t>(sum));
                    if (bad) atomicOr(&flags[r * stride], static_cast<uint32_t>(MI355_STATUS_NONFINITE_ACTIVATION));
                }
            }
        }
        // the row's last quantiser block publishes the row's status word (a row's 32-groups fill whole blocks: hidden % 256 == 0)
        // (the flag words are read-modify-written by device-scope atomics only; the ticket orders them as above)
        const uint32_t r = g0 / groups;
        if constexpr (LINES) {
            // (the A8 image is written by device-scope stores: waves of the same launch, on other XCDs, read it once the row's tag says so)
            if (arrive_last(&ticket[r * stride], groups / 8U)) {
                if (lane == 0) {
                    __hip_atomic_store(&a.status[r], __hip_atomic_load(&flags[r * stride], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(&flags[r * stride], 0U, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                stores_acknowledged();
                if (lane == 0) __hip_atomic_store(row_tag + r, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else {
            __syncthreads();
            if (lane == 0 && __hip_atomic_fetch_add(&ticket[r * stride], 1U, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == groups / 8U - 1U) {
                a.status[r] = __hip_atomic_load(&flags[r * stride], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                flags[r * stride] = 0;
                ticket[r * stride] = 0;
            }
        }
    }
}

// Decode router launch (rows <= 16). Blocks [0, route_blocks) run the logit chains of (row, 8 experts). In the plain form
// (a.plan == nullptr) the kernel stops there. In the fused form blocks [route_blocks, route_blocks + quant_blocks)
// quantise the input rows to A8 (8 groups of 32 per block; the last of a row's blocks publishes the row's status word),
// and the block that finishes a row's last 8 experts (row ticket) runs that row's softmax / top-k / weights and writes the
// row's work items: a decode batch is planned one item per assignment (item i = assignment i, order = identity; the CSR
// fields of the plan are not written), so nothing waits for the other rows. Every ticket word is left zero.
// The place of the code is fixed: the 82 KB of an instance are more than the instruction cache holds, and by where they started - that is, by the
// size of the kernels in front - the same instructions took 18.8 or 20.3 us (8 fp16 rows of hidden 3072, 64 experts; 16 rows 20.3 or 21.7). At a
// multiple of 64 KB | 4 KB, 1, 2, 4, 8, 16 rows: 18.3, 18.9, 17.8, 19.3, 21.6 | 18.8, 19.2, 18.4, 19.2, 20.6.
template <int KIND, bool NORM = false>
__global__ __launch_bounds__(64) __attribute__((aligned(65536))) void route_decode_kernel(RouteArgs a) {
    __shared__ ChainSlot slot0;
    __shared__ ChainSlot slot1;
    __shared__ ChainSlot slot2;
    __shared__ ChainSlot slot3;
    __shared__ uint32_t flag;
    ChainSlot* const slots[4] = {&slot0, &slot1, &slot2, &slot3};
    // the scratch of the select lives in the fourth slot, which is free once the chain has run (every copy into it awaited): LDS per
    // workgroup stays under half a compute unit's, so a
    // launch of more one-wave workgroups than compute units (16 rows x 160 experts: 320) still runs in one round (61 -> 32 us)
    static_assert(sizeof(ChainSlot) >= kRouteMaxExperts * sizeof(float), "select scratch");
    float* const sel_p = reinterpret_cast<float*>(&slot3);
    const uint32_t bid = blockIdx.x, lane = threadIdx.x, neb = (a.p.experts + 7U) / 8U;
    uint32_t* tickets = a.plan ? a.plan + kPlanTicketsAt : nullptr;
    if (bid < a.route_blocks) {
        const uint32_t row = bid / neb;
        route_chain_block<KIND, NORM>(slots, a, row, (bid % neb) * 8U);
        if (!a.plan) return;
        // hand-off between workgroups: the wave's logit stores happen before the barrier, the barrier before lane 0's
        // ticket increment, which releases them at device scope; the workgroup that takes the row's last ticket acquires with
        // the same operation, and its other lanes read the logits after the second barrier
        __syncthreads();
        if (lane == 0) flag = __hip_atomic_fetch_add(&tickets[row], 1U, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == neb - 1U;
        __syncthreads();
        if (flag) {
            if (lane == 0) tickets[row] = 0;
            // The plan of a decode batch. Routed slots: position row * K + slot, one item per assignment. The always-on experts
            // behind them (slot K + s, chosen by every row): positions rows * K + s * rows + row, one item per four rows, so
            // their weights are swept once per four rows and not once per row.
            const uint32_t expert = route_select_row(sel_p, a, row);
            const uint32_t K = a.p.top_k, S = a.p.shared_experts, P = K + S, assignments = a.rows * P, all = a.p.experts + S;
            uint32_t* items = a.plan + plan_items_at(all, assignments);
            uint32_t* order = a.plan + plan_order_at(all);
            if (lane < K) {
                const uint32_t at = row * K + lane;
                *reinterpret_cast<uint4*>(items + 4U * at) = make_uint4(expert, at, at + 1U, row * P + lane + 1U);     // (the item names its assignment)
                order[at] = row * P + lane;
            } else if (lane < P) order[a.rows * K + (lane - K) * a.rows + row] = row * P + lane;
        }
        if (bid == 0) {
            const uint32_t K = a.p.top_k, S = a.p.shared_experts, P = K + S, assignments = a.rows * P, all = a.p.experts + S;
            const uint32_t chunks = (a.rows + 3U) / 4U, made = a.rows * K + S * chunks;
            uint32_t* items = a.plan + plan_items_at(all, assignments);
            if (lane < S * chunks) {
                const uint32_t s_ = lane / chunks, c = lane - s_ * chunks, first = a.rows * K + s_ * a.rows + 4U * c;
                const uint32_t last = 4U * c + 4U < a.rows ? first + 4U : a.rows * K + s_ * a.rows + a.rows;
                *reinterpret_cast<uint4*>(items + 4U * (a.rows * K + lane)) = make_uint4(a.p.experts + s_, first, last, 0U);
            }
            for (uint32_t i = made + lane; i < assignments; i += 64U) *reinterpret_cast<uint4*>(items + 4U * i) = make_uint4(0U, 0U, 0U, 0U);
            if (lane == 0) {
                *a.job_status = 0;
                a.plan[0] = assignments; a.plan[1] = 0; a.plan[2] = S ? 4U : 1U; a.plan[4] = made;
            }
        }
    } else {
        a8_prologue_block<KIND, NORM>(a, bid - a.route_blocks, tickets + 16U, tickets + 128U, 1U);
    }
}

// ======================================================================================================== expert plan
// (layout of the plan words: see the router section above)

// A plan in a launch of its own.
__global__ __launch_bounds__(1024) void plan_kernel(PlanArgs p) {
    __shared__ PlanLds lds;
    plan_block(lds, p, blockIdx.x);
}

// Lanes of the wavefront whose key (of `bits` bits) equals this lane's, among the lanes that `take` part: a ballot per bit.
__device__ __forceinline__ uint64_t lanes_of_key(uint32_t key, uint32_t bits, bool take) {
    uint64_t same = __ballot(take);
    for (uint32_t b = 0; b < bits; ++b) {
        const bool set = (key >> b) & 1U;
        const uint64_t votes = __ballot(set);
        same &= set ? votes : ~votes;
    }
    return same;
}

// The same for at most kPlanSmall assignments, by one workgroup: thread e owns expert e, thread a assignment a. Wave w finds each of its 64 assignments'
// position among its own of the same expert by ballots and leaves the wave's counts; a prefix over the waves and the expert's offset make it the
// position in the order. Bound by latency; alone in its launch it is through before a workgroup per expert has started. A workgroup per expert -> one, 64 |
// 1024 assignments over 128 experts 3.8 | 5.8 -> 3.5 | 4.2 us, over 512 4.6 | 7.8 -> 3.6 | 4.6, over 1024 5.4 | 13.1 -> 4.0 | 5.3; 4096 the other way, 16.2 and 6.0 us.
// (Beside the workgroups of the rows it is the longest one: plan_block.hpp.)
constexpr uint32_t kPlanSmall = 1024;
__global__ __launch_bounds__(1024) void plan_small_kernel(PlanArgs p) {
    __shared__ uint32_t offset[kRouteMaxExperts];
    __shared__ uint16_t wave_counts[16][kRouteMaxExperts];         // per wave and expert, later the prefix over the waves before
    __shared__ u32x4 wave_totals[16];                              // per wave: assignments, items, touched experts, largest group
    const uint32_t tid = threadIdx.x, lane = tid & 63U, wave = tid >> 6, waves = (p.assignments + 63U) / 64U, experts = p.experts;
    for (uint32_t w = 0; w < waves; ++w) wave_counts[w][tid] = 0;
    const uint32_t mine = tid < p.assignments ? p.routes.at(tid) : experts;
    __syncthreads();
    const uint64_t same = lanes_of_key(mine, 32U - static_cast<uint32_t>(__builtin_clz(experts)), mine < experts);
    const uint32_t rank = static_cast<uint32_t>(__popcll(same & ((1ULL << lane) - 1ULL)));
    if (mine < experts && rank == 0) wave_counts[wave][mine] = static_cast<uint16_t>(__popcll(same));
    __syncthreads();
    uint32_t c = 0;
    if (tid < experts)
        for (uint32_t w = 0; w < waves; ++w) {
            const uint32_t here = wave_counts[w][tid];
            wave_counts[w][tid] = static_cast<uint16_t>(c);
            c += here;
        }
    const uint32_t pieces = (c + p.split - 1U) / p.split;
    const uint32_t runs = wave_inclusive_scan(c), items_to = wave_inclusive_scan(pieces), touched_to = static_cast<uint32_t>(__popcll(__ballot(c != 0) & ((2ULL << lane) - 1ULL)));
    uint32_t largest = c;
#pragma unroll
    for (int d = 32; d; d >>= 1) {
        const uint32_t other = __shfl_xor(largest, d);
        largest = other > largest ? other : largest;
    }
    if (lane == 63U) wave_totals[wave] = u32x4{runs, items_to, touched_to, largest};
    __syncthreads();
    u32x4 before = {0U, 0U, 0U, 0U}, all = {0U, 0U, 0U, 0U};
#pragma unroll
    for (uint32_t w = 0; w < 16U; ++w) {
        const u32x4 t = wave_totals[w];
        if (w < wave) { before.x += t.x; before.y += t.y; before.z += t.z; }
        all.x += t.x; all.y += t.y; all.z += t.z; all.w = t.w > all.w ? t.w : all.w;
    }
    const uint32_t first = before.x + runs - c;
    uint32_t* const items = p.plan + plan_items_at(experts, p.assignments);
    if (tid < experts) {
        p.plan[kPlanOffsetsAt + tid] = first;
        if (c != 0) {
            p.plan[plan_touched_at(experts) + before.z + touched_to - 1U] = tid;
            for (uint32_t b = 0, k = before.y + items_to - pieces; b < c; b += p.split, ++k)
                *reinterpret_cast<uint4*>(items + 4U * k) = make_uint4(tid, first + b, first + (b + p.split < c ? b + p.split : c), 0U);
        }
    }
    for (uint32_t u = all.y + tid; u < p.item_bound; u += 1024U) *reinterpret_cast<uint4*>(items + 4U * u) = make_uint4(0U, 0U, 0U, 0U);
    if (tid == 0) {
        p.plan[kPlanOffsetsAt + experts] = all.x;
        p.plan[0] = p.assignments; p.plan[1] = all.z; p.plan[2] = all.w; p.plan[4] = all.y;
    }
    offset[tid] = first;
    __syncthreads();
    if (mine < experts) p.plan[plan_order_at(experts) + offset[mine] + wave_counts[wave][mine] + rank] = tid;
}

// ======================================================================================================== Q4_K x A8 rows
// gate + up + SwiGLU + A8 re-quantisation: one wavefront per (touched expert, 32-output group). Lanes 0..31 hold the
// gate rows of the group, lanes 32..63 the up rows; one cross-half exchange pairs them, then both halves evaluate the
// same 32-value h group.
// Reference: src/cpu/core/routed_expert.cpp:403-427 (gate item), :147-170 (swiglu_quantize).
template <int NA, class IndexOf>
__device__ __forceinline__ void project_epilogue(const float (&value)[NA], const mi355_moe_weights& w, const RowsK& r, uint32_t grp, IndexOf index_of);

// index_of(a): the assignment index of the sweep's activation row a < NA (a may differ between lanes).
template <int NA, int DEPTH, bool NARROW = false, class IndexOf>
__device__ __forceinline__ void project_chunk_of(lds_u8* const (&slots)[DEPTH], const StageSource& source, const mi355_moe_weights& w,
                                                 const RowsK& r, uint32_t grp, IndexOf index_of) {
    const uint32_t lane = threadIdx.x & 63U, o = lane & 31U;
    uint32_t sidx[NA], src[NA], lane_rows[(NA + 3) / 4];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        sidx[a] = __builtin_amdgcn_readfirstlane(index_of(static_cast<uint32_t>(a)));
        src[a] = r.row_of(sidx[a]);
    }
#pragma unroll
    for (int h = 0; h < (NA + 3) / 4; ++h) {
        const uint32_t a = 4U * h + (lane >> 4);
        lane_rows[h] = r.row_of(index_of(a < static_cast<uint32_t>(NA) ? a : 0U));
    }
    const ActRows<NA> act(r.in, src, lane_rows);
    float value[NA];
    sweep_rows<NA, DEPTH, NARROW>(slots, source, w.hidden / 256U, act, value);
    project_epilogue<NA>(value, w, r, grp, index_of);
}

// SwiGLU + A8 re-quantisation of one 32-output group: lanes 0..31 hold the gate values, lanes 32..63 the up values of outputs
// 32 grp .. 32 grp + 31 for each of the NA assignments index_of(0 .. NA - 1). Reference: src/cpu/core/routed_expert.cpp:147-170.
template <int NA, class IndexOf>
__device__ __forceinline__ void project_epilogue(const float (&value)[NA], const mi355_moe_weights& w, const RowsK& r, uint32_t grp, IndexOf index_of) {
    const uint32_t lane = threadIdx.x & 63U, o = lane & 31U;
    uint32_t sidx[NA], src[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        sidx[a] = __builtin_amdgcn_readfirstlane(index_of(static_cast<uint32_t>(a)));
        src[a] = r.row_of(sidx[a]);
    }
    const bool ds = r.awords != nullptr;      // early routes: device-scope stores (an assignment may be written again by a repair)
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        const float other = __shfl_xor(value[a], 32);
        const float g = lane < 32U ? value[a] : other, u = lane < 32U ? other : value[a];
        float gc = g, uc = u;
        swiglu_clamp(gc, uc, w.swiglu_limit);
        const float h = (gc / (1.0F + exp_of(w.exp_kind, -gc))) * uc;
        const uint32_t at_out = grp * 32U + o;
        if (lane < 32U) {
            if (r.gate_out) store_shared_or_plain(ds, r.inter_of(r.gate_out, sidx[a]) + at_out, g);
            if (r.up_out) store_shared_or_plain(ds, r.inter_of(r.up_out, sidx[a]) + at_out, u);
            if (r.h_out) store_shared_or_plain(ds, r.inter_of(r.h_out, sidx[a]) + at_out, h);
        }
        if (!r.h.codes) continue;                         // projection only (the probe form): no A8 image of h
        if (or32_i((finite_f(g) && finite_f(u) && finite_f(h)) ? 0 : 1)) {
            if (lane == 0) {
                if (r.awords) atomicOr(&r.awords[sidx[a]], 0x80000000U);        // early routes: per assignment, folded by the down launch
                else {
                    atomicOr(r.status_of(src[a]), r.nonfinite_bit);
                    atomicOr(r.job_status, static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
                }
            }
        } else {
            const float amax = max32(__builtin_fabsf(h));
            const bool tiny = amax > 0.0F && amax < 0x1p-119F;
            const float dl = (amax == 0.0F || tiny) ? 1.0F : amax / 127.0F;
            const int code = a8_code(h, dl, tiny);
            const int sum = sum32_i(code);
            if (lane < 32U) store_shared_or_plain(ds, r.h_codes_of(sidx[a]) + at_out, static_cast<int8_t>(code));
            if (lane == 0) {
                store_shared_or_plain(ds, r.h_deltas_of(sidx[a]) + grp, dl);
                store_shared_or_plain(ds, r.h_sums_of(sidx[a]) + grp, static_cast<int32_t>(sum));
            }
        }
    }
}

template <int NA, int DEPTH, bool NARROW = false>
__device__ __forceinline__ void project_chunk(lds_u8* const (&slots)[DEPTH], const StageSource& source, const mi355_moe_weights& w,
                                              const RowsK& r, uint32_t grp, uint32_t order_at, uint32_t c0) {
    project_chunk_of<NA, DEPTH, NARROW>(slots, source, w, r, grp, [&](uint32_t a) { return ordered(r, order_at, c0 + a); });
}

#define STRIX_RING_SLOTS(DEPTH, NBMAX)                                                           \
    __shared__ __attribute__((aligned(16))) uint8_t ring0[slot_bytes(NBMAX)];                    \
    __shared__ __attribute__((aligned(16))) uint8_t ring1[slot_bytes(NBMAX)];                    \
    __shared__ __attribute__((aligned(16))) uint8_t ring2[DEPTH > 2 ? slot_bytes(NBMAX) : 16];   \
    __shared__ __attribute__((aligned(16))) uint8_t ring3[DEPTH > 3 ? slot_bytes(NBMAX) : 16];   \
    lds_u8* const ring[4] = {(lds_u8*)ring0, (lds_u8*)ring1, (lds_u8*)ring2, (lds_u8*)ring3};    \
    lds_u8* slots[DEPTH];                                                                        \
    _Pragma("unroll") for (int i = 0; i < DEPTH; ++i) slots[i] = ring[i];

// NBMAX = most activation rows sharing one sweep of the weights (4 for routed experts, 8 for a dense matrix).
template <int NBMAX, int DEPTH>
__global__ __launch_bounds__(64, DEPTH > 3 ? 1 : 2) void project_wave_kernel(mi355_moe_weights w, RowsK r, uint32_t assignments) {
    STRIX_RING_SLOTS(DEPTH, NBMAX)
    const WorkItem item = work_item(w, r, plan_items_at(w.experts, assignments), blockIdx.y);
    const uint32_t e = __builtin_amdgcn_readfirstlane(item.e), begin = __builtin_amdgcn_readfirstlane(item.begin), end = __builtin_amdgcn_readfirstlane(item.end);
    if (begin == end) return;
    // a wave that serves several activation rows has the longest instruction stream of the launch: let it issue first
    if (end - begin > 1U) __builtin_amdgcn_s_setprio(3);
    const uint32_t order_at = plan_order_at(w.experts);
    const uint32_t grp = blockIdx.x;
    const size_t base = static_cast<size_t>(e) * w.gate_expert_stride + static_cast<size_t>(grp * 32U) * w.gate_row_stride;
    const uint8_t* gate = w.gate + base;
    const uint8_t* up = w.up + base;
    const size_t stride = w.gate_row_stride;       // (64-bit: row * stride passes 2^32 for rows of 64 MiB and more)
    StageSource source;
    source.init([&](uint32_t row) { return row < 32U ? gate + row * stride : up + (row - 32U) * stride; });
    lds_u8* const (&sl)[DEPTH] = slots;
    for (uint32_t c0 = begin; c0 < end;) {
        const uint32_t left = end - c0, na = left < static_cast<uint32_t>(NBMAX) ? left : static_cast<uint32_t>(NBMAX);
        switch (na) {
        case 1: project_chunk<1, DEPTH>(sl, source, w, r, grp, order_at, c0); break;
        case 2: project_chunk<2, DEPTH>(sl, source, w, r, grp, order_at, c0); break;
        case 3: project_chunk<3, DEPTH>(sl, source, w, r, grp, order_at, c0); break;
        case 4: project_chunk<4, DEPTH>(sl, source, w, r, grp, order_at, c0); break;
        default:
            if constexpr (NBMAX == 8) {
                switch (na) {
                case 5: project_chunk<5, DEPTH>(sl, source, w, r, grp, order_at, c0); break;
                case 6: project_chunk<6, DEPTH>(sl, source, w, r, grp, order_at, c0); break;
                case 7: project_chunk<7, DEPTH>(sl, source, w, r, grp, order_at, c0); break;
                default: project_chunk<8, DEPTH>(sl, source, w, r, grp, order_at, c0); break;
                }
            }
            break;
        }
        c0 += na;
    }
}

// ---- the front launch of a decode batch planned from early routes (route_early.hpp) ----------------------------------
// One-wave workgroups, in dispatch order:
//   early blocks (row, 4 experts): lane-parallel logits; the block that completes a row picks the row's experts, clears the
//     row's assignment words and publishes one tag {epoch, expert} per assignment;
//   A8 prologue blocks: the A8 image of the input rows; the block that completes a row publishes the row's status word and tag;
//   side blocks (row, 2 experts): the exact logit chains; the block that completes a row runs the exact softmax / top-k / weights
//     (the caller's ids, weights and scores), writes the row's work items (the exact experts: what the down launch reads) and
//     compares its ids with the early ones: where they differ it waits until the assignment's speculative waves have all
//     finished (their count in the assignment's word), clears the word's non-finite flag and recomputes the assignment's h image
//     on the exact expert;
//   projection blocks (assignment, 32-output group): wait for the assignment's tag and the tags of all rows, then one sweep of the
//     tagged expert's gate / up rows; each counts itself into its assignment's word when its part of the h image is acknowledged.
//   helper blocks of a row (experts of many bytes only): wait for the side block's word {epoch, slots}, and sweep every helpers-th group
//     of the slots named there, whose tags name the exact experts by then, in the side block's place.
// Blocks are dispatched in index order, so what a waiting block waits for has been dispatched before it (the repair waits for
// projection blocks, which themselves wait only for blocks in front of them; nothing waits for a helper); every wait is bounded, and a wait that
// runs out (it cannot, short of a lost launch) flags the row as an invalid route: nothing of it is published. Everything that crosses
// workgroups inside the launch - logits, tags, counts, the A8 images of x and of h, the optional fp32 intermediates - moves by
// device-scope stores and loads (an assignment that is repaired is written twice, by waves of different XCDs, and the later
// write has to win at the memory side).
// A waiting wave polls rarely at first and sleeps between polls: a thousand waves polling one line at full rate saturate the
// L2 channel that holds it, and every weight stream crossing that channel with it.
// Two ring slots of 10,240 bytes: eight workgroups share a compute unit.
constexpr uint32_t kFrontSpinLimit = 1U << 22;
struct FrontBlocks { uint32_t early, prologue, side, helpers; };       // helpers: per row
// An assignment whose expert the early choice did not hold (two logits at the edge of the choice within rounding: rare) is swept again, by the side block's one wave while an
// expert's gate and up rows are few, else by helper blocks, kFrontHelpers of them over the rows: one wave takes 0.1 ms a MB. Layers with one such assignment in
// a row, one wave | helpers, us: 1 row of 2048 / 2048 (4.7 MB) 583 | 66, 1, 4 rows of 4096 / 1536 (7 MB) 793, 822 | 76, 129, 1, 6 rows of 6144 / 2560 (18 MB) 1896, 2076 | 156, 464; of
// 2048 / 768 (1.8 MB) 237. Helpers that wait for nothing, none | 64: 1 row of 2048 / 768 25.0 | 25.6, of 4096 / 512 (2.4 MB) 31.3 | 32.3, of 2048 / 2048 39.3 | 39.5, 1, 4 rows of 4096 / 1536
// 47.3, 75.6 | 47.3, 75.8, 1 row of 6144 / 2560 77.1 | 77.0.
constexpr uint64_t kFrontLoneBytes = 4ULL << 20;
constexpr uint32_t kFrontHelpers = 64;
constexpr uint32_t kFrontRunWaves = 86;        // sweeps per super-block of a row past which rows of more than eight of them stream as contiguous stages

// gate + up + SwiGLU + A8 of assignment `at` on expert e, outputs 32 grp .. 32 grp + 31: rows in dense GGUF order whose super-blocks fill a stage's 64 lanes
// (hidden 512, 1024, 2048 and, where the launch's sweeps are enough to be bound by memory, 4096 and 8192) stream as contiguous stages (q4k_blocks.hpp), others as one
// super-block of each row per stage: a contiguous stage of 48 blocks works as long as one of 64, and its chain runs over the lanes in as many steps
// as a row has blocks. Layers, contiguous -> block by block: hidden 1280, 1, 4, 12 rows 30.2, 33.3, 53.7 -> 26.4, 29.6, 44.9 us; 1536 30.5, 34.2 -> 27.2, 31.1; 1792
// 34.6, 41.9 -> 31.8, 39.7; 2304, 1 row 38.3 -> 30.4; 6144, 1 row 97.5 -> 79.3. How many sweeps are enough, contiguous | block by block, rows of hidden / ffn (sweeps):
//   4096: 2 of 1024 (512) 50.8 | 45.7; 3 of 1536 (1152) 68.8 | 66.1; 10 of 512 (1280) 64.8 | 60.3; 5 of 1024 (1280) 75.0 | 73.6; 7 of 768 (1344) 66.2 | 65.8; 11 of 512 (1408) 66.6 |
//   68.4; 6 of 1024 (1536) 78.1 | 80.1; 4 of 1536 (1536) 74.7 | 78.2; 5 of 2560, top-4 (1600) 84.7 | 93.7. 8192: 1 of 2048 (512) 97.3 | 77.0; 6 of 1024 (1536) 144.7 | 140.0; 4 of
//   2048 (2048) 195.2 | 174.8; 5 of 2048 (2560) 230.4 | 223.7; 6 of 2048 (3072) 242.4 | 244.8.
// REPAIR (an assignment that a side block sweeps again, a rare one, by a single wave): block by block whatever the shape, which keeps the registers of the launch's main path.
template <bool REPAIR = false>
__device__ __forceinline__ void front_project(lds_u8* const (&slots)[2], const mi355_moe_weights& w, const RowsK& r, uint32_t e, uint32_t grp, uint32_t at, uint32_t assignments) {
    const size_t base = static_cast<size_t>(e) * w.gate_expert_stride + static_cast<size_t>(grp * 32U) * w.gate_row_stride;
    const uint8_t* gate = w.gate + base;
    const uint8_t* up = w.up + base;
    const uint32_t B = w.hidden / 256U;
    const BlockLanes g = block_lanes(B, 32U);
    const bool runs = g.used == 64U && (B <= 8U || assignments * (w.ffn / 32U) > kFrontRunWaves * B);
    if (!REPAIR && runs && w.gate_row_stride == static_cast<uint64_t>(B) * kQ4kBlock && block_lanes_ok(B, 32U)) {
        const uint32_t half = 32U / g.R;                  // stages of the gate rows, then as many of the up rows
        float value[1];
        const auto stage_base = [&](uint32_t s) { return s < half ? gate + static_cast<size_t>(s) * g.stage_bytes : up + static_cast<size_t>(s - half) * g.stage_bytes; };
        if (g.used == 64U && half == 4U) value[0] = sweep_block_lanes_terms<8>(slots, stage_base, g, r.in, r.row_of(at));      // (hidden 2048)
        else if (g.used == 64U && half == 2U) value[0] = sweep_block_lanes_terms<4>(slots, stage_base, g, r.in, r.row_of(at)); // (hidden 1024)
        else value[0] = sweep_block_lanes<2>(slots, stage_base, 2U * half, g, r.in, r.row_of(at));
        project_epilogue<1>(value, w, r, grp, [&](uint32_t) { return at; });
        return;
    }
    const size_t stride = w.gate_row_stride;
    StageSource source;
    source.init([&](uint32_t q) { return q < 32U ? gate + q * stride : up + (q - 32U) * stride; });
    project_chunk<1, 2>(slots, source, w, r, grp, 0U, at);
}

// The A8 images of every row of the launch are stored. Of every row, not of the one that a sweep reads: deltas and sums of neighbouring rows (hidden / 8 bytes
// each), and code rows of a caller's image that is aligned to 16 bytes only, share cache lines, and the sweep's plain loads bring whole lines into its die's
// L2, where a later sweep of the neighbour would find what it held before. (All lanes; a row's tag per lane, all of them in one line.)
__device__ __forceinline__ bool images_there(const uint32_t* lines, uint32_t rows, uint32_t epoch) {
    const uint32_t lane = threadIdx.x & 63U;
    uint32_t tag = epoch;
    if (lane < rows) tag = __hip_atomic_load(&lines[kLinesRowTags + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __ballot(tag != epoch) == 0;
}

// the word of a row in which its side block tells the row's helpers {epoch, the slots to sweep again}
__device__ __forceinline__ unsigned long long* verdict_of(uint32_t* lines, uint32_t row) { return reinterpret_cast<unsigned long long*>(lines + kLinesVerdict + row * kLineWords); }

template <int KIND, bool HELPED>
__device__ __forceinline__ void side_router_block(lds_u8* const (&slots)[2], const mi355_moe_weights& w, const RowsK& r,
                                                  const RouteArgs& a, uint32_t sb, uint32_t assignments, uint32_t epoch) {
    const uint32_t lane = threadIdx.x & 63U, neb = (a.p.experts + kSideExperts - 1U) / kSideExperts, row = sb / neb;
    side_chain_block<KIND>(slots[0], slots[1], a, row, (sb % neb) * kSideExperts);
    uint32_t* lines = a.plan + kPlanLinesAt;
    if (!arrive_last(&lines[kLinesSide + row * kLineWords], neb)) return;
    const auto tell_helpers = [&](uint32_t again) {
        if (HELPED && lane == 0) __hip_atomic_store(verdict_of(lines, row), (static_cast<unsigned long long>(epoch) << 32) | again, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    const uint32_t expert = route_select_row(reinterpret_cast<float*>((uint8_t*)slots[0]), a, row);
    const uint32_t K = a.p.top_k, P = w.top_k, groups = w.ffn / 32U;          // P: with the always-on slots, which no choice concerns
    if (lane < P) {
        const uint32_t at = row * P + lane;
        *reinterpret_cast<uint4*>(a.plan + plan_items_at(w.experts, assignments) + 4U * at) = make_uint4(expert, at, at + 1U, at + 1U);
        a.plan[plan_order_at(w.experts) + at] = at;
    }
    // the early choice of this row and the A8 images of the input (the repair reads its row's)
    unsigned long long* etags = reinterpret_cast<unsigned long long*>(a.plan + kPlanEtagsAt);
    unsigned long long tag = 0;
    bool there = false;
    for (uint32_t spins = 0; spins < kFrontSpinLimit && !there; ++spins) {
        if (lane < K) tag = __hip_atomic_load(&etags[row * P + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool images = images_there(lines, a.rows, epoch);
        there = __ballot(lane < K && static_cast<uint32_t>(tag >> 32) != epoch) == 0 && images;
        if (!there) __builtin_amdgcn_s_sleep(16);
    }
    asm volatile("" ::: "memory");
    if (!there) {
        if (lane == 0) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_INVALID_ROUTE));
        tell_helpers(0U);
        return;
    }
    uint64_t differ = __ballot(lane < K && static_cast<uint32_t>(tag) != expert);
    // Most differences are the same experts in another order (two scores closer than the early logits resolve): the h image
    // such a slot needs exists already, under the slot that held its expert, and is copied. Only an expert the early choice did not
    // hold at all is swept again. (With the optional fp32 intermediates bound every differing slot is swept again.)
    const uint32_t image_words = w.ffn / 4U + 2U * groups;         // codes, deltas, sums of one assignment, in 32-bit words
    if (differ && !r.gate_out && !r.up_out && !r.h_out) {
        uint32_t src = 0xffU;
        for (uint32_t j = 0; j < K; ++j) {
            const uint32_t held = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(tag)), static_cast<int>(j)));
            if (lane < K && expert == held) src = j;
        }
        uint64_t copy = __ballot(lane < K && ((differ >> lane) & 1ULL) && src != 0xffU);
        if (copy) {
            // every speculative wave of the row has to be through: a slot is read as a source or overwritten as a destination
            bool through = false;
            for (uint32_t spins = 0; spins < kFrontSpinLimit && !through; ++spins) {
                const uint32_t seen = lane < K ? __hip_atomic_load(&r.awords[row * P + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xffffU : groups;
                through = __ballot(seen < groups) == 0;
                if (!through) __builtin_amdgcn_s_sleep(32);
            }
            asm volatile("" ::: "memory");
            if (!through) {
                if (lane == 0) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_INVALID_ROUTE));
                tell_helpers(0U);
                return;
            }
            const auto image_word = [&](uint32_t at, uint32_t i) -> uint32_t* {
                if (i < w.ffn / 4U) return reinterpret_cast<uint32_t*>(r.h_codes_of(at)) + i;
                if (i < w.ffn / 4U + groups) return reinterpret_cast<uint32_t*>(r.h_deltas_of(at)) + (i - w.ffn / 4U);
                return reinterpret_cast<uint32_t*>(r.h_sums_of(at)) + (i - w.ffn / 4U - groups);
            };
            uint32_t* stage = reinterpret_cast<uint32_t*>((uint8_t*)slots[0]);
            uint32_t flags = 0;                                   // bit k: the source of slot k carried the non-finite flag
            for (uint64_t left = copy; left;) {
                const uint32_t k = static_cast<uint32_t>(__ffsll(static_cast<long long>(left))) - 1U;
                left &= left - 1ULL;
                const uint32_t from = row * P + static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(src), static_cast<int>(k)));
                flags |= (__hip_atomic_load(&r.awords[from], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 31) << k;
            }
            // as many words of every image at a time as the ring slot holds; of those all sources first: a source may itself be a destination
            const uint32_t piece = kSideSlotBytes / 4U / K;
            for (uint32_t w0 = 0; w0 < image_words; w0 += piece) {
                const uint32_t n = image_words - w0 < piece ? image_words - w0 : piece;
                for (uint64_t left = copy; left;) {
                    const uint32_t k = static_cast<uint32_t>(__ffsll(static_cast<long long>(left))) - 1U;
                    left &= left - 1ULL;
                    const uint32_t from = row * P + static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(src), static_cast<int>(k)));
                    for (uint32_t i = lane; i < n; i += 64U) stage[k * piece + i] = __hip_atomic_load(image_word(from, w0 + i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                for (uint64_t left = copy; left;) {
                    const uint32_t k = static_cast<uint32_t>(__ffsll(static_cast<long long>(left))) - 1U;
                    left &= left - 1ULL;
                    for (uint32_t i = lane; i < n; i += 64U) __hip_atomic_store(image_word(row * P + k, w0 + i), stage[k * piece + i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            for (uint64_t left = copy; left;) {
                const uint32_t k = static_cast<uint32_t>(__ffsll(static_cast<long long>(left))) - 1U;
                left &= left - 1ULL;
                if (lane == 0) __hip_atomic_store(&r.awords[row * P + k], groups | (((flags >> k) & 1U) << 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");      // the staged images are out of LDS before a sweep reuses the slot
            differ &= ~copy;
        }
    }
    uint32_t again = 0;
    while (differ) {
        const uint32_t k = static_cast<uint32_t>(__ffsll(static_cast<long long>(differ))) - 1U;
        differ &= differ - 1ULL;
        const uint32_t at = row * P + k, e = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(expert), static_cast<int>(k)));
        uint32_t seen = 0;
        for (uint32_t spins = 0; spins < kFrontSpinLimit; ++spins) {
            seen = __hip_atomic_load(&r.awords[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xffffU;
            if (seen >= groups) break;
            __builtin_amdgcn_s_sleep(32);
        }
        asm volatile("" ::: "memory");
        if (seen < groups) {
            if (lane == 0) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_INVALID_ROUTE));
            continue;
        }
        if (lane == 0) __hip_atomic_store(&r.awords[at], groups, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if constexpr (HELPED) {
            if (lane == 0) __hip_atomic_store(&etags[at], (static_cast<unsigned long long>(epoch) << 32) | e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            again |= 1U << k;
        } else {
            for (uint32_t grp = 0; grp < groups; ++grp) front_project<true>(slots, w, r, e, grp, at, assignments);
        }
    }
    if (again) stores_acknowledged();
    tell_helpers(again);
}

// One of a row's helpers: waits for the side block's word and sweeps its share of the slots named there, every helpers-th of their groups.
__device__ __forceinline__ void front_helper_block(lds_u8* const (&slots)[2], const mi355_moe_weights& w, const RowsK& r, uint32_t* plan, uint32_t row, uint32_t helper,
                                                   uint32_t helpers, uint32_t assignments, uint32_t epoch) {
    unsigned long long word = 0;
    for (uint32_t spins = 0; spins < kFrontSpinLimit && static_cast<uint32_t>(word >> 32) != epoch; ++spins) {
        if (spins == 0) __builtin_amdgcn_s_sleep(127); else __builtin_amdgcn_s_sleep(2);
        word = __hip_atomic_load(verdict_of(plan + kPlanLinesAt, row), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("" ::: "memory");
    if (static_cast<uint32_t>(word >> 32) != epoch) {
        if ((threadIdx.x & 63U) == 0) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_INVALID_ROUTE));
        return;
    }
    const unsigned long long* etags = reinterpret_cast<const unsigned long long*>(plan + kPlanEtagsAt);
    const uint32_t groups = w.ffn / 32U;
    uint32_t grp = helper;
    for (uint32_t left = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(word)); left; left &= left - 1U) {
        const uint32_t at = row * w.top_k + static_cast<uint32_t>(__builtin_ctz(left));
        const uint32_t e = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(__hip_atomic_load(&etags[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)));
        for (; grp < groups; grp += helpers) front_project<true>(slots, w, r, e, grp, at, assignments);
        grp -= groups;
    }
}

template <int KIND, bool HELPED>
__global__ __launch_bounds__(64, 2) void layer_front_kernel(mi355_moe_weights w, RowsK views, uint32_t assignments, RouteArgs a, FrontBlocks nb) {
    const RowsK r = dense_views(views);
    // exactly 20,480 bytes of LDS: eight workgroups fill a compute unit's 160 KB (one more byte and only seven fit)
    __shared__ __attribute__((aligned(16))) uint8_t ring0[kSideSlotBytes];
    __shared__ __attribute__((aligned(16))) uint8_t ring1[kSideSlotBytes];
    static_assert(kSideSlotBytes == slot_bytes(4), "the projection sweep's slot");
    lds_u8* const slots[2] = {(lds_u8*)ring0, (lds_u8*)ring1};
    lds_u8* const (&sl)[2] = slots;
    uint32_t bid = blockIdx.x;
    const uint32_t lane = threadIdx.x, K = a.p.top_k, P = w.top_k;      // P: with the always-on slots (experts behind the routed ones)
    uint32_t* lines = a.plan + kPlanLinesAt;
    const uint32_t epoch = lines[kLinesEpoch] + 1U;                 // (stored back by the down launch of this call)
    unsigned long long* etags = reinterpret_cast<unsigned long long*>(a.plan + kPlanEtagsAt);
    if (bid < nb.early) {
        const uint32_t neb = (a.p.experts + kEarlyExperts - 1U) / kEarlyExperts, row = bid / neb;
        // the row's first early block also selects: it clears the row's assignment words before anything else (acknowledged long before
        // its tags go out), brings its own four logits, then reads the row's logits until every one carries this call's epoch
        const bool selects = bid % neb == 0;
        if (selects && lane < P) __hip_atomic_store(&r.awords[row * P + lane], 0U, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        early_logits_block<KIND>(a, row, (bid % neb) * kEarlyExperts, epoch);
        if (bid == 0 && lane == 0) {
            *a.job_status = 0;
            a.plan[0] = assignments; a.plan[1] = 0; a.plan[2] = 1U; a.plan[4] = assignments;
        }
        if (!selects) return;
        bool ok;
        const uint32_t chosen = early_select_row(a, row, epoch, ok), expert = lane < K ? chosen : a.p.experts + (lane - K);
        if (!ok) {
            if (lane == 0) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_INVALID_ROUTE));
            return;
        }
        stores_acknowledged();
        if (lane < P) __hip_atomic_store(&etags[row * P + lane], (static_cast<unsigned long long>(epoch) << 32) | expert, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    bid -= nb.early;
    if (bid < nb.prologue) {
        a8_prologue_block<KIND, false, true>(a, bid, lines + kLinesPrologue, lines + kLinesPrologue + 1U, kLineWords, lines + kLinesRowTags, epoch);
        return;
    }
    bid -= nb.prologue;
    if (bid < nb.side) {
        side_router_block<KIND, HELPED>(sl, w, r, a, bid, assignments, epoch);
        return;
    }
    bid -= nb.side;
    if (HELPED && bid >= assignments * (w.ffn / 32U)) {
        bid -= assignments * (w.ffn / 32U);
        front_helper_block(sl, w, r, a.plan, bid / nb.helpers, bid % nb.helpers, nb.helpers, assignments, epoch);
        return;
    }
    // Projection block: assignment `at`, 32-output group `grp`. (Sharing one sweep among the rows that chose an expert was
    // measured slower: the sweeps that serve several rows finish last, and the others do not speed up.)
    const uint32_t groups = w.ffn / 32U, at = bid / groups, grp = bid - at * groups, row = at / P;
    unsigned long long tag = 0;
    bool there = false;
    for (uint32_t spins = 0; spins < kFrontSpinLimit && !there; ++spins) {
        tag = __hip_atomic_load(&etags[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool images = images_there(lines, a.rows, epoch);
        there = static_cast<uint32_t>(tag >> 32) == epoch && images;
        // a block that finds nothing at its first look started with the launch: the tags are microseconds away (one long sleep,
        // about 3 us); a block dispatched later, into a freed slot, finds them at once
        if (!there) { if (spins == 0) __builtin_amdgcn_s_sleep(127); else __builtin_amdgcn_s_sleep(8); }
    }
    asm volatile("" ::: "memory");
    if (!there) {
        if (lane == 0) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_INVALID_ROUTE));
        return;
    }
    const uint32_t e = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(tag))));
    // The compute unit issues its oldest waves first, so the blocks dispatched last fall behind the others stage by stage and the
    // launch ends with a few hundred of them alone on the memory system: the later a block's place in the dispatch, the higher
    // its issue priority (the launch at 8 rows: 0.3 - 0.5 us).
    {
        const uint32_t quarter = bid * 4U / (assignments * groups);
        if (quarter == 1U) __builtin_amdgcn_s_setprio(1);
        else if (quarter == 2U) __builtin_amdgcn_s_setprio(2);
        else if (quarter == 3U) __builtin_amdgcn_s_setprio(3);
    }
    front_project(sl, w, r, e, grp, at, assignments);
    stores_acknowledged();
    if (lane == 0) __hip_atomic_fetch_add(&r.awords[at], 1U, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// down rows: one wavefront per (touched expert, 64 hidden outputs), lane = output row.
// Reference: src/cpu/core/routed_expert.cpp:429-447 (down item), src/moe_a8_down_contract.cpp:146 (Q4_K down row).
template <int NA, int DEPTH>
__device__ __forceinline__ void down_chunk(lds_u8* const (&slots)[DEPTH], const StageSource& source, const mi355_moe_weights& w,
                                           const RowsK& r, uint32_t order_at, uint32_t c0) {
    uint32_t src[NA], lane_rows[(NA + 3) / 4];
#pragma unroll
    for (int a = 0; a < NA; ++a) src[a] = __builtin_amdgcn_readfirstlane(ordered(r, order_at, c0 + a));
#pragma unroll
    for (int h = 0; h < (NA + 3) / 4; ++h) {
        const uint32_t a = 4U * h + ((threadIdx.x & 63U) >> 4);
        lane_rows[h] = ordered(r, order_at, c0 + (a < static_cast<uint32_t>(NA) ? a : 0U));
    }
    const ActRows<NA> act(r.h, src, lane_rows);
    float value[NA];
    sweep_rows<NA, DEPTH>(slots, source, w.ffn / 256U, act, value);
    const uint32_t o = blockIdx.x * 64U + (threadIdx.x & 63U);
#pragma unroll
    for (int a = 0; a < NA; ++a) r.rawdots_of(src[a], w.hidden)[o] = value[a];
}

template <int NBMAX, int DEPTH>
__global__ __launch_bounds__(64, DEPTH > 3 ? 1 : 2) void down_wave_kernel(mi355_moe_weights w, RowsK r, uint32_t assignments) {
    STRIX_RING_SLOTS(DEPTH, NBMAX)
    const WorkItem item = work_item(w, r, plan_items_at(w.experts, assignments), blockIdx.y);
    const uint32_t e = __builtin_amdgcn_readfirstlane(item.e), begin = __builtin_amdgcn_readfirstlane(item.begin), end = __builtin_amdgcn_readfirstlane(item.end);
    if (begin == end) return;
    if (*r.job_status & MI355_STATUS_NONFINITE_PROJECTION) return;
    if (end - begin > 1U) __builtin_amdgcn_s_setprio(3);     // as in the projection: the longest instruction streams issue first
    const uint32_t order_at = plan_order_at(w.experts);
    const uint8_t* rows = w.down + static_cast<size_t>(e) * w.down_expert_stride + static_cast<size_t>(blockIdx.x * 64U) * w.down_row_stride;
    const size_t stride = w.down_row_stride;
    StageSource source;
    source.init([&](uint32_t row) { return rows + row * stride; });
    lds_u8* const (&sl)[DEPTH] = slots;
    for (uint32_t c0 = begin; c0 < end;) {
        const uint32_t left = end - c0, na = left < static_cast<uint32_t>(NBMAX) ? left : static_cast<uint32_t>(NBMAX);
        switch (na) {
        case 1: down_chunk<1, DEPTH>(sl, source, w, r, order_at, c0); break;
        case 2: down_chunk<2, DEPTH>(sl, source, w, r, order_at, c0); break;
        case 3: down_chunk<3, DEPTH>(sl, source, w, r, order_at, c0); break;
        case 4: down_chunk<4, DEPTH>(sl, source, w, r, order_at, c0); break;
        default:
            if constexpr (NBMAX == 8) {
                switch (na) {
                case 5: down_chunk<5, DEPTH>(sl, source, w, r, order_at, c0); break;
                case 6: down_chunk<6, DEPTH>(sl, source, w, r, order_at, c0); break;
                case 7: down_chunk<7, DEPTH>(sl, source, w, r, order_at, c0); break;
                default: down_chunk<8, DEPTH>(sl, source, w, r, order_at, c0); break;
                }
            }
            break;
        }
        c0 += na;
    }
}


// ---- the smallest decode batches: 16 rows per wavefront, lane = (row, pair) (q4k_quads.hpp) ------------------------------
#define STRIX_QUAD_SLOTS(DEPTH)                                                                      \
    __shared__ __attribute__((aligned(16))) uint8_t quad0[4][kQuadSlotBytes];                         \
    __shared__ __attribute__((aligned(16))) uint8_t quad1[4][kQuadSlotBytes];                         \
    __shared__ __attribute__((aligned(16))) uint8_t quad2[DEPTH > 2 ? 4 : 1][DEPTH > 2 ? kQuadSlotBytes : 16]; \
    __shared__ __attribute__((aligned(16))) uint8_t quad3[DEPTH > 3 ? 4 : 1][DEPTH > 3 ? kQuadSlotBytes : 16]; \
    const uint32_t wave = threadIdx.x >> 6;                                                           \
    lds_u8* const quad_ring[4] = {(lds_u8*)quad0[wave], (lds_u8*)quad1[wave], (lds_u8*)quad2[DEPTH > 2 ? wave : 0], (lds_u8*)quad3[DEPTH > 3 ? wave : 0]}; \
    lds_u8* slots[DEPTH];                                                                             \
    _Pragma("unroll") for (int i = 0; i < DEPTH; ++i) slots[i] = quad_ring[i];

// gate + up + SwiGLU + A8 of one item (one assignment): a 4-wave workgroup per 32-output group, wave = 8 gate rows and the
// 8 up rows of the same features. Reference: src/cpu/core/routed_expert.cpp:403-427, :147-170.
template <int DEPTH>
__global__ __launch_bounds__(256) void project_quad_kernel(mi355_moe_weights w, RowsK r, uint32_t assignments) {
    STRIX_QUAD_SLOTS(DEPTH)
    __shared__ float wg_amax[4];
    __shared__ int wg_sum[4], wg_bad[4];
    const WorkItem item = work_item(w, r, plan_items_at(w.experts, assignments), blockIdx.y);
    const uint32_t e = item.e, begin = item.begin, end = item.end;
    if (begin == end) return;
    const uint32_t lane = threadIdx.x & 63U, p = lane & 3U, rr = lane >> 2, grp = blockIdx.x;
    const uint32_t sidx = __builtin_amdgcn_readfirstlane(ordered(r, plan_order_at(w.experts), begin)), row = r.row_of(sidx);
    const uint32_t f0 = grp * 32U + 8U * wave;
    const size_t base = static_cast<size_t>(e) * w.gate_expert_stride + static_cast<size_t>(f0) * w.gate_row_stride;
    const uint8_t* gate = w.gate + base;
    const uint8_t* up = w.up + base;
    const size_t stride = w.gate_row_stride;
    QuadSource source;
    source.init([&](uint32_t q) { return q < 8U ? gate + q * stride : up + (q - 8U) * stride; }, r.in.codes_of(row));
    lds_u8* const (&sl)[DEPTH] = slots;
    const float value = sweep_quads<DEPTH>(sl, source, w.hidden / 256U, r.in, row);
    const float other = __shfl_xor(value, 32);
    const bool mine = lane < 32U && p == 0;                   // the lane that publishes feature f0 + rr
    const float g = lane < 32U ? value : other, u = lane < 32U ? other : value;
    float gc = g, uc = u;
    swiglu_clamp(gc, uc, w.swiglu_limit);
    const float h = (gc / (1.0F + exp_of(w.exp_kind, -gc))) * uc;
    const uint32_t at_out = f0 + rr;
    if (mine) {
        if (r.gate_out) r.inter_of(r.gate_out, sidx)[at_out] = g;
        if (r.up_out) r.inter_of(r.up_out, sidx)[at_out] = u;
        if (r.h_out) r.inter_of(r.h_out, sidx)[at_out] = h;
    }
    if (!r.h.codes) return;                               // projection only (the probe form): no A8 image of h
    const int bad = or32_i((mine && !(finite_f(g) && finite_f(u) && finite_f(h))) ? 1 : 0);
    const float amax_wave = max32(mine ? __builtin_fabsf(h) : 0.0F);
    if (lane == 0) { wg_amax[wave] = amax_wave; wg_bad[wave] = bad; }
    __syncthreads();
    if (wg_bad[0] | wg_bad[1] | wg_bad[2] | wg_bad[3]) {
        if (threadIdx.x == 0) {
            atomicOr(r.status_of(row), r.nonfinite_bit);
            atomicOr(r.job_status, static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
        }
        return;
    }
    const float amax = __builtin_fmaxf(__builtin_fmaxf(wg_amax[0], wg_amax[1]), __builtin_fmaxf(wg_amax[2], wg_amax[3]));
    const bool tiny = amax > 0.0F && amax < 0x1p-119F;
    const float dl = (amax == 0.0F || tiny) ? 1.0F : amax / 127.0F;
    const int code = a8_code(h, dl, tiny);
    const int sum_wave = sum32_i(mine ? code : 0);
    if (lane == 0) wg_sum[wave] = sum_wave;
    if (mine) r.h_codes_of(sidx)[at_out] = static_cast<int8_t>(code);
    __syncthreads();
    if (threadIdx.x == 0) {
        r.h_deltas_of(sidx)[grp] = dl;
        r.h_sums_of(sidx)[grp] = wg_sum[0] + wg_sum[1] + wg_sum[2] + wg_sum[3];
    }
}

// The same for Q5_K gate / up tensors (176-byte blocks through the same ring), for every assignment of the item in turn.
template <int DEPTH>
__global__ __launch_bounds__(256) void project_q5k_kernel(mi355_moe_weights w, RowsK r, uint32_t assignments) {
    STRIX_QUAD_SLOTS(DEPTH)
    __shared__ float wg_amax[4];
    __shared__ int wg_sum[4], wg_bad[4];
    const WorkItem item = work_item(w, r, plan_items_at(w.experts, assignments), blockIdx.y);
    const uint32_t e = item.e, begin = item.begin, end = item.end;
    const uint32_t lane = threadIdx.x & 63U, p = lane & 3U, rr = lane >> 2, grp = blockIdx.x;
    const uint32_t f0 = grp * 32U + 8U * wave;
    const size_t base = static_cast<size_t>(e) * w.gate_expert_stride + static_cast<size_t>(f0) * w.gate_row_stride;
    const uint8_t* gate = w.gate + base;
    const uint8_t* up = w.up + base;
    const size_t stride = w.gate_row_stride;
    lds_u8* const (&sl)[DEPTH] = slots;
    const bool mine = lane < 32U && p == 0;                   // the lane that publishes feature f0 + rr
    for (uint32_t a = begin; a < end; ++a) {
        const uint32_t sidx = __builtin_amdgcn_readfirstlane(ordered(r, plan_order_at(w.experts), a)), row = r.row_of(sidx);
        QuadSourceT<11> source;
        source.init([&](uint32_t q) { return q < 8U ? gate + q * stride : up + (q - 8U) * stride; }, r.in.codes_of(row));
        const float value = sweep_quads<DEPTH, true>(sl, source, w.hidden / 256U, r.in, row);
        const float other = __shfl_xor(value, 32);
        const float g = lane < 32U ? value : other, u = lane < 32U ? other : value;
        float gc = g, uc = u;
        swiglu_clamp(gc, uc, w.swiglu_limit);
        const float h = (gc / (1.0F + exp_of(w.exp_kind, -gc))) * uc;
        const uint32_t at_out = f0 + rr;
        if (mine) {
            if (r.gate_out) r.inter_of(r.gate_out, sidx)[at_out] = g;
            if (r.up_out) r.inter_of(r.up_out, sidx)[at_out] = u;
            if (r.h_out) r.inter_of(r.h_out, sidx)[at_out] = h;
        }
        if (!r.h.codes) continue;                         // projection only (the probe form): no A8 image of h
        const int bad = or32_i((mine && !(finite_f(g) && finite_f(u) && finite_f(h))) ? 1 : 0);
        const float amax_wave = max32(mine ? __builtin_fabsf(h) : 0.0F);
        __syncthreads();                                          // the previous assignment's reads of the shared words are done
        if (lane == 0) { wg_amax[wave] = amax_wave; wg_bad[wave] = bad; }
        __syncthreads();
        if (wg_bad[0] | wg_bad[1] | wg_bad[2] | wg_bad[3]) {      // uniform over the workgroup
            if (threadIdx.x == 0) {
                atomicOr(r.status_of(row), r.nonfinite_bit);
                atomicOr(r.job_status, static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
            }
            continue;
        }
        const float amax = __builtin_fmaxf(__builtin_fmaxf(wg_amax[0], wg_amax[1]), __builtin_fmaxf(wg_amax[2], wg_amax[3]));
        const bool tiny = amax > 0.0F && amax < 0x1p-119F;
        const float dl = (amax == 0.0F || tiny) ? 1.0F : amax / 127.0F;
        const int code = a8_code(h, dl, tiny);
        const int sum_wave = sum32_i(mine ? code : 0);
        if (lane == 0) wg_sum[wave] = sum_wave;
        if (mine) r.h_codes_of(sidx)[at_out] = static_cast<int8_t>(code);
        __syncthreads();
        if (threadIdx.x == 0) {
            r.h_deltas_of(sidx)[grp] = dl;
            r.h_sums_of(sidx)[grp] = wg_sum[0] + wg_sum[1] + wg_sum[2] + wg_sum[3];
        }
    }
}

// down rows of one item: a 4-wave workgroup per 64 outputs, 16 per wave.
// Reference: src/cpu/core/routed_expert.cpp:429-447, src/moe_a8_down_contract.cpp:146.
template <int DEPTH>
__global__ __launch_bounds__(256) void down_quad_kernel(mi355_moe_weights w, RowsK r, uint32_t assignments) {
    STRIX_QUAD_SLOTS(DEPTH)
    const WorkItem item = work_item(w, r, plan_items_at(w.experts, assignments), blockIdx.y);
    const uint32_t e = item.e, begin = item.begin, end = item.end;
    if (begin == end) return;
    if (*r.job_status & MI355_STATUS_NONFINITE_PROJECTION) return;
    const uint32_t lane = threadIdx.x & 63U, p = lane & 3U, rr = lane >> 2;
    const uint32_t src = __builtin_amdgcn_readfirstlane(ordered(r, plan_order_at(w.experts), begin));
    const uint32_t o0 = blockIdx.x * 64U + 16U * wave;
    const uint8_t* rows = w.down + static_cast<size_t>(e) * w.down_expert_stride + static_cast<size_t>(o0) * w.down_row_stride;
    const size_t stride = w.down_row_stride;
    QuadSource source;
    source.init([&](uint32_t q) { return rows + q * stride; }, r.h.codes_of(src));
    lds_u8* const (&sl)[DEPTH] = slots;
    const float value = sweep_quads<DEPTH>(sl, source, w.ffn / 256U, r.h, src);
    if (p == 0) r.rawdots_of(src, w.hidden)[o0 + rr] = value;
}

// Ordered combine of the slots of one row. Reference: include/strix/moe/combine.hpp:36-59 (fma form),
// src/ds41_expert_tp.cpp:189-199 (product then add, slots in ascending expert id).
// VEC = columns per thread (4: every row of rawdots / base / output starts on 16 bytes and hidden % 4 == 0). The slots'
// values are all requested before the chain starts, so a thread has top_k loads in flight instead of one.
// Bound by latency up to some hundred rows. So every wavefront looks the row up by itself - lane k the route and weight of slot k, its place
// in the ascending order by comparison with the others' - and in slot order nothing stands in front of the values' loads: one way to memory
// (two in ascending order), where one thread of the workgroup, a barrier and, for the order, an insertion sort over routes in memory took
// up to four (16 rows x 6144, top-8 ascending: 8.4 -> 5.0 us; 333 rows x 2048, top-8 11.2 -> 6.3; 1000 rows 18.8 -> 13.0).
template <int VEC>
__global__ __launch_bounds__(256) void merge_kernel(mi355_moe_weights w, RowsK r, uint32_t form) {
    typedef float vec_t __attribute__((ext_vector_type(VEC)));
    const uint32_t row = blockIdx.y, o = (blockIdx.x * 256U + threadIdx.x) * VEC, lane = threadIdx.x & 63U, K = w.top_k;
    // fail closed: a row flagged by an earlier stage publishes nothing (the aggregate bit is this kernel's own), and
    // neither does any row of a job whose down phase was skipped (its unweighted outputs are not this job's)
    const uint32_t row_status = *r.status_of(row), job = *r.job_status;
    const bool ascending = form == MI355_COMBINE_MULADD_ASCENDING_EXPERT;
    const float weight = lane < K ? r.route_weights_of(row)[lane] : 0.0F;
    const uint32_t at = o < w.hidden ? o : 0U;
    const float* const values = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(r.rawdots) + row * r.rawdots_rs) + at;
    vec_t e[16];
    uint32_t slot[16];
    if (!ascending) {
#pragma unroll
        for (uint32_t k = 0; k < 16U; ++k) slot[k] = k;
    } else {
        const uint32_t route = lane < K ? r.routes_of(row)[lane] : 0xffffffffU;
        uint32_t place = 0;                               // stable: an equal expert in an earlier slot goes first
#pragma unroll
        for (uint32_t k = 0; k < 16U; ++k) {
            const uint32_t other = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(route), static_cast<int>(k)));
            place += k < K && (other < route || (other == route && k < lane)) ? 1U : 0U;
        }
#pragma unroll
        for (uint32_t k = 0; k < 16U; ++k) slot[k] = k < K ? static_cast<uint32_t>(__builtin_ctzll(__ballot(lane < K && place == k))) : 0U;
    }
#pragma unroll
    for (uint32_t k = 0; k < 16U; ++k)
        if (k < K) e[k] = *reinterpret_cast<const vec_t*>(values + static_cast<size_t>(slot[k]) * w.hidden);
    if (o >= w.hidden || (row_status & ~static_cast<uint32_t>(MI355_STATUS_AGGREGATE)) || (job & MI355_STATUS_NONFINITE_PROJECTION)) return;
    vec_t y;
    bool finite = true;
    float acc[VEC];
#pragma unroll
    for (int c = 0; c < VEC; ++c) acc[c] = 0.0F;
#pragma unroll
    for (uint32_t k = 0; k < 16U; ++k) {
        if (k >= K) continue;
        const float wt = f_of(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(b_of(weight)), static_cast<int>(slot[k]))));
#pragma unroll
        for (int c = 0; c < VEC; ++c) {
            if (!ascending && k + r.shared_slots < K) acc[c] = __builtin_fmaf(wt, e[k][c], acc[c]);
            else acc[c] = acc[c] + wt * e[k][c];
        }
    }
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
        const float out = r.base ? acc[c] + r.base_of(row)[o + c] : acc[c];
        finite = finite && finite_f(out);
        y[c] = out;
    }
    if (!finite) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_AGGREGATE));
    *reinterpret_cast<vec_t*>(r.output + static_cast<size_t>(row) * r.output_stride + o) = y;
}

constexpr uint32_t kDownMergeSlots = 8;        // top_k bound: 8 waves x 2 ring slots fill the LDS of a compute unit
constexpr uint32_t kDownMergeMost = 16;        // of the forms of 16 columns, whose slots are smaller or none (instances of 8, 9 - top-8 and an always-on expert - and 16)
// What a down + combine launch looks up at its start, in this order and without a branch between the requests: its item, the job word and what
// the fold needs. The sweep waits for the item; asked for behind the others, or behind branches whose arguments are fetched one block after
// the other, it stood a way to memory further back. The launch, fold behind the barrier by one thread | requests in front of the item |
// behind it: Q4_K, hidden 3072 / ffn 768 / 64 experts top-8, 1, 4 rows 5.8, 12.4 | 6.1, 13.1 | 6.1, 12.6 us, hidden 4096 / ffn 1280, top-4, 8
// rows 26.2 | 24.7 | 23.9; hidden 2048 / ffn 768 / 128 experts top-8, 16 rows, Q6_K 40.4 | 40.8 | 39.4, Q8_0 38.2 | 36.8 | 36.7, Q5_1 30.2 | 31.0 | 29.4.
//
// the item of (row, slot): the fused router plans one per assignment, in assignment order
__device__ __forceinline__ WorkItem slot_item(const mi355_moe_weights& w, const RowsK& r, uint32_t assignments, uint32_t a) {
    const uint4 item = *reinterpret_cast<const uint4*>(r.plan + plan_items_at(w.experts, assignments) + 4U * a);
    __builtin_amdgcn_sched_barrier(0);
    return {item.x, item.y, item.z, item.w};
}
// The job word. A batch planned from early routes (r.awords): the front launch left its non-finite flags per assignment; every workgroup
// folds them to the same job word, the first workgroup of a row publishes its row's.
struct DownJob { uint32_t word[2]; };
__device__ __forceinline__ DownJob down_job_request(const RowsK& r, uint32_t assignments, uint32_t lane) {
    const uint32_t* const words = r.awords ? r.awords : r.job_status;
    const uint32_t last = r.awords ? assignments - 1U : 0U;
    return DownJob{{words[lane < last ? lane : last], words[lane + 64U < last ? lane + 64U : last]}};       // (past the last one: the last one again)
}
__device__ __forceinline__ uint32_t down_job(const DownJob& d, const mi355_moe_weights& w, const RowsK& r, uint32_t row, uint32_t wave, uint32_t lane) {
    if (!r.awords) return __builtin_amdgcn_readfirstlane(d.word[0]);
    const uint32_t job = (__ballot(d.word[0] >> 31) | __ballot(d.word[1] >> 31)) ? static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION) : 0U;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) r.plan[kPlanLinesAt + kLinesEpoch] += 1U;      // this call's epoch is spent
    if (job && blockIdx.x == 0 && wave == 0) {
        const uint32_t lo = row * w.top_k, hi = lo + w.top_k;
        const bool mine = (lane >= lo && lane < hi && (d.word[0] >> 31)) || (lane + 64U >= lo && lane + 64U < hi && (d.word[1] >> 31));
        const bool any = __ballot(mine) != 0;
        if (lane == 0) {
            if (any) atomicOr(r.status_of(row), r.nonfinite_bit);
            atomicOr(r.job_status, static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
        }
    }
    return job;
}
// What the fold of a row's slots needs beside their values (lane k: weight and expert of slot k; the row's status as the launches before left
// it, by a vector load; the base of column o - without one any word, which nothing reads).
struct SlotFold { float weight, base; uint32_t route, status; };
__device__ __forceinline__ SlotFold slot_fold_request(const mi355_moe_weights& w, const RowsK& r, uint32_t row, uint32_t o, uint32_t lane) {
    const uint32_t k = lane < w.top_k ? lane : 0U;
    const float* const base = r.base ? r.base_of(row) + o : r.route_weights_of(row);
    SlotFold f;
    f.status = __hip_atomic_load(r.status_of(row), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    f.weight = r.route_weights_of(row)[k];
    f.route = r.routes_of(row)[k];
    f.base = *base;
    return f;
}
// The row's value of one column, as merge_kernel folds it (every lane of the wavefront takes part). Fail closed: a row flagged by an
// earlier stage publishes nothing (the aggregate bit is the combine's own).
template <uint32_t SLOTS, class Value>
__device__ __forceinline__ void slot_fold(const SlotFold& f, const mi355_moe_weights& w, const RowsK& r, uint32_t row, uint32_t o, uint32_t form, bool stores, uint32_t lane, Value value) {
    if (f.status & ~static_cast<uint32_t>(MI355_STATUS_AGGREGATE)) return;
    const uint32_t K = w.top_k;
    const bool ascending = form == MI355_COMBINE_MULADD_ASCENDING_EXPERT;
    uint32_t place = lane;                                   // of the lane's slot; stable: an equal expert in an earlier slot goes first
    if (ascending) {
        place = 0;
#pragma unroll
        for (uint32_t k = 0; k < SLOTS; ++k) {
            const uint32_t other = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(f.route), static_cast<int>(k)));
            place += k < K && (other < f.route || (other == f.route && k < lane)) ? 1U : 0U;
        }
    }
    float acc = 0.0F;
#pragma unroll
    for (uint32_t k = 0; k < SLOTS; ++k) {
        if (k >= K) continue;
        const uint32_t slot = ascending ? static_cast<uint32_t>(__builtin_ctzll(__ballot(lane < K && place == k))) : k;
        const float wt = f_of(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(b_of(f.weight)), static_cast<int>(slot)))), ev = value(slot);
        if (!ascending && k + r.shared_slots < K) acc = __builtin_fmaf(wt, ev, acc);
        else acc = acc + wt * ev;
    }
    if (!stores) return;
    const float y = r.base ? acc + f.base : acc;
    if (!finite_f(y)) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_AGGREGATE));
    r.output[static_cast<size_t>(row) * r.output_stride + o] = y;
}

// Down rows and the ordered combine of a decode batch in one launch: a workgroup owns (row, 64 output columns) and has one
// wave per slot of the row, wave k sweeping the down rows of the expert in slot k (the plan holds one item per assignment,
// in assignment order); the waves leave their 64 values in LDS and wave 0 folds them exactly as merge_kernel does. Only
// waves of one workgroup exchange data, so nothing depends on the visibility of another workgroup's stores.
// Reference: src/cpu/core/routed_expert.cpp:429-447, src/moe_a8_down_contract.cpp:146, include/strix/moe/combine.hpp:36-59.
__global__ __launch_bounds__(64 * kDownMergeSlots) void down_merge_kernel(mi355_moe_weights w, RowsK views, uint32_t assignments, uint32_t form) {
    const RowsK r = dense_views(views);
    // the two ring slots are separate LDS objects: the compiler then knows that a copy into one never touches the other and lets
    // the reads of the landed slot go ahead while the next stage's copy is in flight (as slots of one array it waited for both)
    __shared__ __attribute__((aligned(16))) uint8_t ring_even[kDownMergeSlots][slot_bytes(1)];
    __shared__ __attribute__((aligned(16))) uint8_t ring_odd[kDownMergeSlots][slot_bytes(1)];
    __shared__ float slot_value[kDownMergeSlots][64];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63U, row = blockIdx.y, o = blockIdx.x * 64U + lane;
    const uint32_t a = row * w.top_k + wave;
    const WorkItem item = slot_item(w, r, assignments, a);
    const DownJob job = down_job_request(r, assignments, lane);                // (requested together with the item: one round trip, not two)
    const SlotFold fold = slot_fold_request(w, r, row, o, lane);
    const uint32_t e = __builtin_amdgcn_readfirstlane(item.e), begin = __builtin_amdgcn_readfirstlane(item.begin), end = __builtin_amdgcn_readfirstlane(item.end);
    if (down_job(job, w, r, row, wave, lane) & MI355_STATUS_NONFINITE_PROJECTION) return;                       // the whole job: no down rows, nothing published
    float value = 0.0F;
    if (begin != end) {                                                        // (an invalid route has no item: its row is flagged)
        const uint32_t first = item.first ? item.first - 1U : ordered(r, plan_order_at(w.experts), begin);
        const uint8_t* rows = w.down + static_cast<size_t>(e) * w.down_expert_stride + static_cast<size_t>(blockIdx.x * 64U) * w.down_row_stride;
        const size_t stride = w.down_row_stride;
        lds_u8* const slots[2] = {(lds_u8*)ring_even[wave], (lds_u8*)ring_odd[wave]};
        const uint32_t src[1] = {static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(first))}, lane_rows[1] = {first};
        // (contiguous stages - q4k_blocks.hpp - would be four of 16 rows here instead of three of 64: a wave's time is its number of
        // stage waits, and that form measured 16.9 us against 15.5)
        StageSource source;
        source.init([&](uint32_t q) { return rows + q * stride; });
        const ActRows<1> act(r.h, src, lane_rows);
        float swept[1];
        sweep_rows<1, 2, true>(slots, source, w.ffn / 256U, act, swept);      // narrow codes copies: the slots are slot_bytes(1)
        value = swept[0];
        r.rawdots_of(src[0], w.hidden)[o] = value;
    }
    slot_value[wave][lane] = value;
    __syncthreads();
    if (wave == 0) slot_fold<kDownMergeSlots>(fold, w, r, row, o, form, true, lane, [&](uint32_t slot) { return slot_value[slot][lane]; });
}

// down_merge_kernel for dense rows of at most four super-blocks (down_row_stride = B * 144): the 64 rows of a column block stream as B
// contiguous stages of 1 KB pieces instead of B stages of 64 separate 144-byte blocks (a read-only launch of this shape moves the
// same bytes in 11.8 us against 14.4 us), the block terms meet in LDS in block order and lane = row adds them in ascending order.
// (Fold behind the barrier: asked for at the start, in front of the item, 1, 8, 16 rows of hidden 2048 / ffn 768 27.7, 45.9, 73.5 -> 28.2, 46.2, 73.9 us.)
template <int B>
__global__ __launch_bounds__(64 * kDownMergeSlots) void down_merge_flat_kernel(mi355_moe_weights w, RowsK views, uint32_t assignments, uint32_t form) {
    const RowsK r = dense_views(views);
    // (the two ring slots are separate LDS objects, as in down_merge_kernel)
    __shared__ __attribute__((aligned(16))) uint8_t ring_even[kDownMergeSlots][kFlatStageBytes];
    __shared__ __attribute__((aligned(16))) uint8_t ring_odd[kDownMergeSlots][kFlatStageBytes];
    __shared__ __attribute__((aligned(16))) uint8_t act_rows[kDownMergeSlots][flat_act_bytes(B)];
    __shared__ float slot_value[kDownMergeSlots][64];
    __shared__ uint32_t slot_order[kDownMergeSlots];
    __shared__ float slot_weight[kDownMergeSlots];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63U, row = blockIdx.y, o = blockIdx.x * 64U + lane;
    uint32_t job;                                                              // (requested together with the item: one round trip, not two)
    uint32_t word[2] = {0U, 0U};
    if (r.awords) {
        if (lane < assignments) word[0] = r.awords[lane];
        if (lane + 64U < assignments) word[1] = r.awords[lane + 64U];
    } else job = *r.job_status;
    const uint32_t a = row * w.top_k + wave;
    const WorkItem item = work_item(w, r, plan_items_at(w.experts, assignments), a);
    const uint32_t e = __builtin_amdgcn_readfirstlane(item.e), begin = __builtin_amdgcn_readfirstlane(item.begin), end = __builtin_amdgcn_readfirstlane(item.end);
    if (r.awords) {
        // a batch planned from early routes: the front launch left its non-finite flags per assignment; every workgroup folds them
        // to the same job word, the first workgroup of a row publishes its row's
        job = (__ballot(word[0] >> 31) | __ballot(word[1] >> 31)) ? static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION) : 0U;
        if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) r.plan[kPlanLinesAt + kLinesEpoch] += 1U;      // this call's epoch is spent
        if (job && blockIdx.x == 0 && wave == 0) {
            const uint32_t lo = row * w.top_k, hi = lo + w.top_k;
            const bool mine = (lane >= lo && lane < hi && (word[0] >> 31)) || (lane + 64U >= lo && lane + 64U < hi && (word[1] >> 31));
            const bool any = __ballot(mine) != 0;
            if (lane == 0) {
                if (any) atomicOr(r.status_of(row), r.nonfinite_bit);
                atomicOr(r.job_status, static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
            }
        }
    }
    if (job & MI355_STATUS_NONFINITE_PROJECTION) return;                       // the whole job: no down rows, nothing published
    float value = 0.0F;
    if (begin != end) {                                                        // (an invalid route has no item: its row is flagged)
        const uint32_t first = item.first ? item.first - 1U : ordered(r, plan_order_at(w.experts), begin);
        // the 64 rows of the column block are one run of 64 * B super-blocks: B contiguous stages (q4k_blocks.hpp)
        const uint8_t* rows = w.down + static_cast<size_t>(e) * w.down_expert_stride + static_cast<size_t>(blockIdx.x * 64U) * w.down_row_stride;
        lds_u8* const slots[2] = {(lds_u8*)ring_even[wave], (lds_u8*)ring_odd[wave]};
        const uint32_t src[1] = {static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(first))};
        value = sweep_flat_rows<B, 2>(slots, (lds_u8*)act_rows[wave], rows, r.h, src[0]);
        r.rawdots_of(src[0], w.hidden)[o] = value;
    }
    slot_value[wave][lane] = value;
    if (threadIdx.x == 0) {
        for (uint32_t k = 0; k < w.top_k; ++k) slot_order[k] = k;
        if (form == MI355_COMBINE_MULADD_ASCENDING_EXPERT)
            for (uint32_t i = 1; i < w.top_k; ++i)
                for (uint32_t j = i; j > 0 && r.routes_of(row)[slot_order[j]] < r.routes_of(row)[slot_order[j - 1]]; --j) {
                    const uint32_t t = slot_order[j]; slot_order[j] = slot_order[j - 1]; slot_order[j - 1] = t;
                }
        for (uint32_t k = 0; k < w.top_k; ++k) slot_weight[k] = r.route_weights_of(row)[slot_order[k]];
    }
    __syncthreads();
    // fail closed: a row flagged by an earlier stage publishes nothing (the aggregate bit is the combine's own)
    if (wave != 0 || (*r.status_of(row) & ~static_cast<uint32_t>(MI355_STATUS_AGGREGATE))) return;
    float acc = 0.0F;
    for (uint32_t k = 0; k < w.top_k; ++k) {
        const float ev = slot_value[slot_order[k]][lane];
        if (form == MI355_COMBINE_FMA_SLOT_ORDER && k + r.shared_slots < w.top_k) acc = __builtin_fmaf(slot_weight[k], ev, acc);
        else acc = acc + slot_weight[k] * ev;
    }
    const float y = r.base ? acc + r.base_of(row)[o] : acc;
    if (!finite_f(y)) atomicOr(r.status_of(row), static_cast<uint32_t>(MI355_STATUS_AGGREGATE));
    r.output[static_cast<size_t>(row) * r.output_stride + o] = y;
}


// The same for the smallest decode batches, in the 16-rows-per-wavefront layout of down_quad_kernel: a workgroup owns (row, 16
// output columns), wave k sweeps the 16 down rows of the expert in slot k (lane = (row, pair)), the slots' values meet in LDS
// and the first sixteen lanes of wave 0 fold them as merge_kernel does. One launch instead of two for one to six rows.
template <int DEPTH, uint32_t SLOTS>
__global__ __launch_bounds__(64 * SLOTS) void down_merge_quad_kernel(mi355_moe_weights w, RowsK views, uint32_t assignments, uint32_t form) {
    const RowsK r = dense_views(views);
    __shared__ __attribute__((aligned(16))) uint8_t mq0[SLOTS][kQuadSlotBytes];
    __shared__ __attribute__((aligned(16))) uint8_t mq1[SLOTS][kQuadSlotBytes];
    __shared__ __attribute__((aligned(16))) uint8_t mq2[DEPTH > 2 ? SLOTS : 1][DEPTH > 2 ? kQuadSlotBytes : 16];
    __shared__ __attribute__((aligned(16))) uint8_t mq3[DEPTH > 3 ? SLOTS : 1][DEPTH > 3 ? kQuadSlotBytes : 16];
    __shared__ float slot_value[SLOTS][kQuadRows];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63U, p = lane & 3U, rr = lane >> 2, row = blockIdx.y, o0 = blockIdx.x * kQuadRows;
    lds_u8* const ring[4] = {(lds_u8*)mq0[wave], (lds_u8*)mq1[wave], (lds_u8*)mq2[DEPTH > 2 ? wave : 0], (lds_u8*)mq3[DEPTH > 3 ? wave : 0]};
    lds_u8* slots[DEPTH];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) slots[i] = ring[i];
    const uint32_t oc = blockIdx.x * 16U + (lane & 15U);                       // the folding lane's column
    const uint32_t a = row * w.top_k + wave;
    const WorkItem item = slot_item(w, r, assignments, a);
    const DownJob job = down_job_request(r, assignments, lane);                // (requested together with the item)
    const SlotFold fold = slot_fold_request(w, r, row, oc, lane);
    if (down_job(job, w, r, row, wave, lane) & MI355_STATUS_NONFINITE_PROJECTION) return;                       // the whole job: no down rows, nothing published
    float value = 0.0F;
    if (item.begin != item.end) {                                              // (an invalid route has no item: its row is flagged)
        const uint32_t src = __builtin_amdgcn_readfirstlane(item.first ? item.first - 1U : ordered(r, plan_order_at(w.experts), item.begin));
        const uint8_t* rows = w.down + static_cast<size_t>(item.e) * w.down_expert_stride + static_cast<size_t>(o0) * w.down_row_stride;
        const size_t stride = w.down_row_stride;
        QuadSource source;
        source.init([&](uint32_t q) { return rows + q * stride; }, r.h.codes_of(src));
        lds_u8* const (&sl)[DEPTH] = slots;
        value = sweep_quads<DEPTH>(sl, source, w.ffn / 256U, r.h, src);
        if (p == 0) r.rawdots_of(src, w.hidden)[o0 + rr] = value;
    }
    if (p == 0) slot_value[wave][rr] = value;
    __syncthreads();
    if (wave == 0) slot_fold<SLOTS>(fold, w, r, row, oc, form, lane < 16U, lane, [&](uint32_t slot) { return slot_value[slot][lane & 15U]; });
}

// Down rows + combine in one launch for Q5_1 down rows of whole, 16-byte aligned super-blocks (the host executor's format,
// src/cpu/core/routed_expert.cpp:110-126): the workgroup of (row, 16 columns), wave k = the expert in slot k, each wave with
// the copy ring, the lane layout and the chain order of down_q51_ring_kernel for its one assignment.
template <int DEPTH, uint32_t SLOTS>
__global__ __launch_bounds__(64 * SLOTS) void down_merge_q51_kernel(mi355_moe_weights w, RowsK views, uint32_t assignments, uint32_t form) {
    const RowsK r = dense_views(views);
    typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
    typedef const __attribute__((address_space(3))) float lds_f32c;
    typedef const __attribute__((address_space(3))) int32_t lds_i32c;
    constexpr uint32_t kBlock = kQ51Block, RP = group_row_pieces(), WC = group_weight_copies(), PER = WC + 2U;
    // a slot: the 16 rows' 8 groups (3 KB), the one assignment's 256 codes and its [8 deltas][8 sums]
    constexpr uint32_t ROWB = kGroupStage * kBlock, CODES_AT = 1024U * WC, TABLE_AT = CODES_AT + 256U, SLOT = TABLE_AT + 64U;
    static_assert(16U * ROWB == 1024U * WC, "the rows of a stage fill the weight copies");
    __shared__ __attribute__((aligned(16))) uint8_t ring_mem[DEPTH][SLOTS][SLOT];
    __shared__ float slot_value[SLOTS][16];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63U, j = lane & 3U, rr = lane >> 2, row = blockIdx.y;
    const uint32_t o0 = blockIdx.x * 16U, o = o0 + rr;
    const uint32_t oc = blockIdx.x * 16U + (lane & 15U);                       // the folding lane's column
    const WorkItem item = slot_item(w, r, assignments, row * w.top_k + wave);
    const DownJob job = down_job_request(r, assignments, lane);                // (requested together with the item)
    const SlotFold fold = slot_fold_request(w, r, row, oc, lane);
    if (down_job(job, w, r, row, wave, lane) & MI355_STATUS_NONFINITE_PROJECTION) return;                       // the whole job: no down rows, nothing published
    float value = 0.0F;
    if (item.begin != item.end) {                                              // (an invalid route has no item: its row is flagged)
        const uint32_t src = item.first ? item.first - 1U : ordered(r, plan_order_at(w.experts), item.begin);
        const uint32_t stages = w.ffn / 256U;
        const uint8_t* rows = w.down + static_cast<size_t>(item.e) * w.down_expert_stride + static_cast<size_t>(o0) * w.down_row_stride;
        // the lane's pieces of a stage: piece index i * 64 + lane = row * RP + piece of the row's 8-group segment
        const uint8_t* wsrc[WC];
#pragma unroll
        for (uint32_t i = 0; i < WC; ++i) {
            uint32_t k = i * 64U + lane;
            k = k < 16U * RP ? k : 16U * RP - 1U;                  // padding lanes repeat the last piece into unused LDS
            const uint32_t wr = k / RP, piece = k - RP * wr;
            wsrc[i] = rows + static_cast<size_t>(wr) * w.down_row_stride + 16U * piece;
        }
        // the stage's 256 codes (lanes 0..15) and its [8 deltas][8 sums] (lanes 0..3)
        const uint8_t* csrc = reinterpret_cast<const uint8_t*>(r.h.codes_of(src)) + 16U * (lane & 15U);
        const uint32_t tq = lane & 3U;
        const uint8_t* tsrc = tq < 2U ? reinterpret_cast<const uint8_t*>(r.h.deltas_of(src)) + 16U * tq : reinterpret_cast<const uint8_t*>(r.h.sums_of(src)) + 16U * (tq - 2U);
        const auto start = [&](lds_u8* slot) {
#pragma unroll
            for (uint32_t i = 0; i < WC; ++i) {
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)wsrc[i],
                                                 (__attribute__((address_space(3))) void*)(slot + 1024U * i), 16, 0, 0);
                wsrc[i] += ROWB;
            }
            if (lane < 16U)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)csrc,
                                                 (__attribute__((address_space(3))) void*)(slot + CODES_AT), 16, 0, 0);
            csrc += 256;
            if (lane < 4U)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)tsrc,
                                                 (__attribute__((address_space(3))) void*)(slot + TABLE_AT), 16, 0, 0);
            tsrc += 32;
        };
        lds_u8* ring[DEPTH];
#pragma unroll
        for (int s = 0; s < DEPTH; ++s) ring[s] = (lds_u8*)ring_mem[s][wave];
        float chain = 0.0F;
#pragma unroll
        for (int s = 0; s < DEPTH - 1; ++s)
            if (static_cast<uint32_t>(s) < stages) start(ring[s]);
        for (uint32_t b0 = 0; b0 < stages; b0 += DEPTH) {
#pragma unroll
            for (int s = 0; s < DEPTH; ++s) {
                const uint32_t b = b0 + s;
                if (b < stages) {
                    const uint32_t last = b + DEPTH - 1U < stages ? b + DEPTH - 1U : stages;
                    wait_stages_ahead<PER>(last - 1U - b);
                    if (b + DEPTH - 1U < stages) start(ring[(s + DEPTH - 1) % DEPTH]);
                    const lds_u8* slot = ring[s];
#pragma unroll
                    for (uint32_t c = 0; c < kGroupStage / 4U; ++c) {
                        const uint32_t gl = 4U * c + j;                                 // the lane's group inside the stage
                        float d, m;
                        uint32_t q[8];
                        load_q51_block_lds(slot + rr * ROWB + gl * kBlock, d, m, q);
                        lds_u32x4* codes = (lds_u32x4*)(slot + CODES_AT + 32U * gl);
                        const u32x4 c_lo = codes[0], c_hi = codes[1];
                        const uint32_t cw[8] = {c_lo.x, c_lo.y, c_lo.z, c_lo.w, c_hi.x, c_hi.y, c_hi.z, c_hi.w};
                        int dot = 0;
#pragma unroll
                        for (int i = 0; i < 8; ++i) dot = __builtin_amdgcn_sdot4(static_cast<int>(q[i]), static_cast<int>(cw[i]), dot, false);
                        const float first = d * static_cast<float>(dot);
                        const float combined = first + (m * static_cast<float>(*(lds_i32c*)(slot + TABLE_AT + 32U + 4U * gl)));
                        chain = chain + (*(lds_f32c*)(slot + TABLE_AT + 4U * gl) * combined);
                    }
                }
            }
        }
        value = chain;
        value = value + xor1_f(value);          // chain0 + chain1 | chain2 + chain3
        value = value + xor2_f(value);          // (chain0 + chain1) + (chain2 + chain3)
        if (j == 0) r.rawdots_of(src, w.hidden)[o] = value;
    }
    if (j == 0) slot_value[wave][rr] = value;
    __syncthreads();
    if (wave == 0) slot_fold<SLOTS>(fold, w, r, row, oc, form, lane < 16U, lane, [&](uint32_t slot) { return slot_value[slot][lane & 15U]; });
}

// Down rows + combine in one launch for Q6_K down rows (src/moe_a8_down_contract.cpp:147-158): the workgroup of (row, 16 columns),
// wave k = the expert in slot k, lane = (row, pair) with the direct loads and the order of down_q6k_kernel. Bound by its loads (q6k_part); three blocks' worth of them
// asked for together (a bound on the registers, for a workgroup more on a compute unit, costs more than it gives: 8, 16 rows 55.8, 88.6 us). Layers of hidden 2048 /
// ffn 768 / 128 experts top-8, 1, 8, 16 rows 25.7, 57.8, 92.1 -> 25.1, 54.3, 85.9 us; 5 of them with the norm and an always-on expert 57.3 -> 52.0; 4 rows of 4096 /
// 1536 / 64 103.4 -> 94.2; 6 rows of 3072 / 2304 / 32 top-4 100.6 -> 87.8.
template <uint32_t SLOTS>
__global__ __launch_bounds__(64 * SLOTS) void down_merge_q6k_kernel(mi355_moe_weights w, RowsK views, uint32_t assignments, uint32_t form) {
    const RowsK r = dense_views(views);
    __shared__ float slot_value[SLOTS][16];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63U, p = lane & 3U, half = p >> 1, odd = p & 1U, rr = lane >> 2, row = blockIdx.y;
    const uint32_t o = blockIdx.x * 16U + rr;
    const uint32_t oc = blockIdx.x * 16U + (lane & 15U);                       // the folding lane's column
    const WorkItem item = slot_item(w, r, assignments, row * w.top_k + wave);
    const DownJob job = down_job_request(r, assignments, lane);                // (requested together with the item)
    const SlotFold fold = slot_fold_request(w, r, row, oc, lane);
    if (down_job(job, w, r, row, wave, lane) & MI355_STATUS_NONFINITE_PROJECTION) return;                       // the whole job: no down rows, nothing published
    float value = 0.0F;
    if (item.begin != item.end) {                                              // (an invalid route has no item: its row is flagged)
        const uint32_t src = item.first ? item.first - 1U : ordered(r, plan_order_at(w.experts), item.begin);
        const uint32_t blocks = w.ffn / 256U;
        const uint8_t* wrow = w.down + static_cast<size_t>(item.e) * w.down_expert_stride + static_cast<size_t>(o) * w.down_row_stride;
        const int8_t* h_codes = r.h.codes_of(src);
        const float* h_deltas = r.h.deltas_of(src);
        float acc = 0.0F;
#pragma unroll 3
        for (uint32_t b = 0; b < blocks; ++b) {
            Q6kPart part;
            q6k_part(part, wrow + static_cast<size_t>(b) * kQ6kBlock, half, odd);
            acc = acc + q6k_part_term(part, h_codes + 256U * b, h_deltas + 8U * b, half, odd);
        }
        value = acc;
        value = value + xor1_f(value);          // acc0 + acc1 | acc2 + acc3
        value = value + xor2_f(value);          // (acc0 + acc1) + (acc2 + acc3)
        if (p == 0) r.rawdots_of(src, w.hidden)[o] = value;
    }
    if (p == 0) slot_value[wave][rr] = value;
    __syncthreads();
    if (wave == 0) slot_fold<SLOTS>(fold, w, r, row, oc, form, lane < 16U, lane, [&](uint32_t slot) { return slot_value[slot][lane & 15U]; });
}

// Down rows + combine in one launch for Q8_0 down tensors (the host executor's format, src/cpu/core/routed_expert.cpp:110-126): the
// workgroup of (row, 16 columns) again, wave k = the expert in slot k, lane = (row, chain) with the direct block loads and the
// chain order of down_groups_kernel<0>; one item per assignment (the fused decode router's plan).
// (The image of h by global loads - from a pointer that may come out of a table they were flat ones, which wait for the LDS as well -, three groups of a chain's asked
// for together, two in the wider workgroups: 8, 16 rows of 2048 / 768 / 128 57.5, 90.1 -> 56.3, 88.7 us, 4 of 4096 / 1536 / 64 98.9 -> 96.6.)
template <uint32_t SLOTS>
__global__ __launch_bounds__(64 * SLOTS) void down_merge_q8_0_kernel(mi355_moe_weights w, RowsK views, uint32_t assignments, uint32_t form) {
    const RowsK r = dense_views(views);
    typedef uint32_t u32x4_g __attribute__((ext_vector_type(4)));
    __shared__ float slot_value[SLOTS][16];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63U, j = lane & 3U, odd = j & 1U, rr = lane >> 2, row = blockIdx.y;
    const uint32_t o = blockIdx.x * 16U + rr;
    const uint32_t oc = blockIdx.x * 16U + (lane & 15U);                       // the folding lane's column
    const WorkItem item = slot_item(w, r, assignments, row * w.top_k + wave);
    const DownJob job = down_job_request(r, assignments, lane);                // (requested together with the item)
    const SlotFold fold = slot_fold_request(w, r, row, oc, lane);
    if (down_job(job, w, r, row, wave, lane) & MI355_STATUS_NONFINITE_PROJECTION) return;                       // the whole job: no down rows, nothing published
    float value = 0.0F;
    if (item.begin != item.end) {                                              // (an invalid route has no item: its row is flagged)
        const uint32_t src = item.first ? item.first - 1U : ordered(r, plan_order_at(w.experts), item.begin);
        const uint32_t per_chain = w.ffn / 128U;
        const uint8_t* wrow = w.down + static_cast<size_t>(item.e) * w.down_expert_stride + static_cast<size_t>(o) * w.down_row_stride + 34U * j;
        const int8_t* h_codes = r.h.codes_of(src);
        const float* h_deltas = r.h.deltas_of(src);
        float chain = 0.0F;
#pragma unroll (SLOTS > kDownMergeSlots ? 2 : 3)
        for (uint32_t c = 0; c < per_chain; ++c) {
            const uint32_t g = 4U * c + j;
            float d, m;
            uint32_t q[8];
            load_group_block<0>(wrow + static_cast<size_t>(c) * (4U * 34U), odd, d, m, q);
            const auto* codes = in_global<u32x4_g>(h_codes + 32U * g);
            const u32x4_g c_lo = codes[0], c_hi = codes[1];
            const uint32_t cw[8] = {c_lo.x, c_lo.y, c_lo.z, c_lo.w, c_hi.x, c_hi.y, c_hi.z, c_hi.w};
            int dot = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) dot = __builtin_amdgcn_sdot4(static_cast<int>(q[i]), static_cast<int>(cw[i]), dot, false);
            chain = chain + (in_global<float>(h_deltas)[g] * (d * static_cast<float>(dot)));
        }
        value = chain;
        value = value + xor1_f(value);          // chain0 + chain1 | chain2 + chain3
        value = value + xor2_f(value);          // (chain0 + chain1) + (chain2 + chain3)
        if (j == 0) r.rawdots_of(src, w.hidden)[o] = value;
    }
    if (j == 0) slot_value[wave][rr] = value;
    __syncthreads();
    if (wave == 0) slot_fold<SLOTS>(fold, w, r, row, oc, form, lane < 16U, lane, [&](uint32_t slot) { return slot_value[slot][lane & 15U]; });
}

// SwiGLU + A8 re-quantisation of dense gate/up rows. Reference: src/cpu/core/routed_expert.cpp:147-170.
__global__ __launch_bounds__(256) void swiglu_quantize_kernel(const float* gate, const float* up, uint32_t ffn, uint32_t exp_kind, float limit,
                                                              int8_t* codes, float* deltas, int32_t* sums, float* h_out, uint32_t* status,
                                                              uint32_t* job_status) {
    const uint32_t row = blockIdx.y, groups = ffn / 32U, grp = blockIdx.x * 8U + (threadIdx.x >> 5), l = threadIdx.x & 31U;
    if (grp >= groups) return;
    const size_t at = static_cast<size_t>(row) * ffn + grp * 32U + l;
    const float g = gate[at], u = up[at];
    float gc = g, uc = u;
    swiglu_clamp(gc, uc, limit);
    const float ex = exp_of(exp_kind, -gc);
    const float hv = (gc / (1.0F + ex)) * uc;
    if (h_out) h_out[at] = hv;
    const int bad = or32_i((finite_f(g) && finite_f(u) && finite_f(hv)) ? 0 : 1);
    if (bad) {
        if (l == 0 && status) atomicOr(&status[row], static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
        if (l == 0 && job_status) atomicOr(job_status, static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
        return;
    }
    const float amax = max32(__builtin_fabsf(hv));
    const bool tiny = amax > 0.0F && amax < 0x1p-119F;
    const float dl = (amax == 0.0F || tiny) ? 1.0F : amax / 127.0F;
    const int code = a8_code(hv, dl, tiny);
    const int sum = sum32_i(code);
    codes[at] = static_cast<int8_t>(code);
    if (l == 0) {
        deltas[static_cast<size_t>(row) * groups + grp] = dl;
        sums[static_cast<size_t>(row) * groups + grp] = sum;
    }
}

// ======================================================================================================== dispatch
// Up to 4 (routed experts) or 8 (dense matrix) activation rows share one sweep of an expert's weights; an expert with
// more assignments is swept again for the rest.
// Ring depth: the deepest of 4, 3, 2 at which every workgroup of the launch is resident at once (LDS is what limits it).
inline int ring_depth(uint64_t waves, int nbmax) {
    for (int d = 4; d > 2; --d)
        if (waves <= resident_waves(static_cast<uint32_t>(d) * slot_bytes(nbmax))) return d;
    return 2;
}
template <int NBMAX>
inline void launch_project_nb(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, dim3 grid, hipStream_t st) {
    switch (ring_depth(static_cast<uint64_t>(grid.x) * grid.y, NBMAX)) {
    case 4: project_wave_kernel<NBMAX, 4><<<grid, 64, 0, st>>>(w, r, rows * w.top_k); break;
    case 3: project_wave_kernel<NBMAX, 3><<<grid, 64, 0, st>>>(w, r, rows * w.top_k); break;
    default: project_wave_kernel<NBMAX, 2><<<grid, 64, 0, st>>>(w, r, rows * w.top_k); break;
    }
}
template <int NBMAX>
inline void launch_down_nb(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, dim3 grid, hipStream_t st) {
    switch (ring_depth(static_cast<uint64_t>(grid.x) * grid.y, NBMAX)) {
    case 4: down_wave_kernel<NBMAX, 4><<<grid, 64, 0, st>>>(w, r, rows * w.top_k); break;
    case 3: down_wave_kernel<NBMAX, 3><<<grid, 64, 0, st>>>(w, r, rows * w.top_k); break;
    default: down_wave_kernel<NBMAX, 2><<<grid, 64, 0, st>>>(w, r, rows * w.top_k); break;
    }
}
inline RowsK rows_k(const mi355_moe_rows& r, const mi355_moe_weights& w) {
    RowsK k{};
    static_cast<mi355_moe_rows&>(k) = r;
    k.slot_stride = w.ffn;
    k.top_k = w.top_k;
    k.nonfinite_bit = MI355_STATUS_NONFINITE_PROJECTION;
    k.in = dense_image(r.codes, r.deltas, r.sums, w.hidden);
    k.h = dense_image(r.down_codes, r.down_deltas, r.down_sums, w.ffn);
    k.routes_rs = k.route_weights_rs = 4ULL * w.top_k;
    k.status_rs = 4;
    k.inter_rs = 4ULL * w.top_k * w.ffn;
    k.rawdots_rs = 4ULL * w.top_k * w.hidden;
    k.base_rs = 4ULL * w.hidden;
    return k;
}
// every per-row view back to back (the layouts of mi355_moe_rows): the forms that read the fields as plain arrays apply
inline bool dense_rows(const RowsK& k, const mi355_moe_weights& w) {
    return !k.assignments && !k.in.table && k.in.per_row == 1U && k.in.codes_rs == w.hidden && k.in.deltas_rs == w.hidden / 8U && k.in.sums_rs == w.hidden / 8U &&
           k.h.per_row == 1U && k.h.codes_rs == w.ffn && k.h.deltas_rs == w.ffn / 8U && k.h.sums_rs == w.ffn / 8U && k.slot_stride == w.ffn &&
           k.inter_rs == 4ULL * w.top_k * w.ffn && k.rawdots_rs == 4ULL * w.top_k * w.hidden && k.status_rs == 4;
}

// ---- dense matrix (one expert, every row uses it): the pair-per-lane sweep ------------------------------------------
template <int NA, int AL, int KL = 1>
inline void launch_pairs_depth(const PairArgs& a, uint32_t matrices, hipStream_t st) {
    const dim3 grid(a.rows / pair_rows<AL, KL>(), matrices);
    const uint64_t waves = static_cast<uint64_t>(grid.x) * grid.y;
    // 4 slots when every wavefront of the launch is resident with them and the wait counter can express 3 stages ahead
    const bool deep = 3U * pair_copies<NA, AL, KL>() <= 63U && waves <= resident_waves(4U * pair_slot_bytes<NA, AL, KL>());
    if (deep) q4k_pairs_kernel<NA, AL, 4, KL><<<grid, 64, 0, st>>>(a);
    else q4k_pairs_kernel<NA, AL, 2, KL><<<grid, 64, 0, st>>>(a);
}
// nacts <= 8 activation rows. A matrix with few rows gives few wavefronts, each with a long instruction stream (the whole
// of K): such launches spread every row over more lanes - the four super-blocks of a stage over a quad and, with >= 4
// activation rows, two activation lanes - which multiplies the wavefronts and divides each one's instruction stream.
inline void launch_pairs(const PairArgs& a, uint32_t matrices, hipStream_t st) {
    const bool narrow = static_cast<uint64_t>(a.rows) * matrices < 16384U;
    if (a.nacts <= 1U) { if (narrow) launch_pairs_depth<1, 1, 4>(a, matrices, st); else launch_pairs_depth<1, 1>(a, matrices, st); }
    else if (a.nacts <= 2U) { if (narrow) launch_pairs_depth<2, 1, 4>(a, matrices, st); else launch_pairs_depth<2, 1>(a, matrices, st); }
    else if (a.nacts <= 4U) { if (narrow) launch_pairs_depth<2, 2, 4>(a, matrices, st); else launch_pairs_depth<4, 1>(a, matrices, st); }
    else { if (narrow) launch_pairs_depth<4, 2, 4>(a, matrices, st); else launch_pairs_depth<8, 1>(a, matrices, st); }
}
// The dense form needs fp32 gate / up rows as workspace (the optional intermediates views) because a wavefront holds
// 16 rows, not a whole 32-output SwiGLU group.
inline bool dense_pairs_ok(const mi355_moe_weights& w, uint32_t rows) {
    return w.gate_type == MI355_TYPE_Q4_K && w.down_type == MI355_TYPE_Q4_K &&
           w.experts == 1U && w.top_k == 1U && rows <= 8U && (w.hidden / 256U) % kPairBlocks == 0 && (w.ffn / 256U) % kPairBlocks == 0 &&
           w.gate_row_stride < (1ULL << 24) && w.down_row_stride < (1ULL << 24);
}
inline void launch_project_dense(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, hipStream_t st) {
    PairArgs a{};
    a.m[0] = PairMatrix{w.gate, w.gate_row_stride, r.gate_out, w.ffn};
    a.m[1] = PairMatrix{w.up, w.gate_row_stride, r.up_out, w.ffn};
    a.rows = w.ffn; a.blocks = w.hidden / 256U; a.img = r.in; a.nacts = rows;
    launch_pairs(a, 2, st);
    swiglu_quantize_kernel<<<dim3((w.ffn / 32U + 7U) / 8U, rows), 256, 0, st>>>(r.gate_out, r.up_out, w.ffn, w.exp_kind, w.swiglu_limit, r.down_codes, r.down_deltas,
                                                                                r.down_sums, r.h_out, r.status, r.job_status);
}
inline void launch_down_dense(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, hipStream_t st) {
    PairArgs a{};
    a.m[0] = PairMatrix{w.down, w.down_row_stride, r.rawdots, w.hidden};
    a.rows = w.hidden; a.blocks = w.ffn / 256U; a.img = r.h; a.nacts = rows;
    a.skip_flag = r.job_status; a.skip_mask = MI355_STATUS_NONFINITE_PROJECTION;
    a.publish = r;                 // (r.top1_form != 0: the launch publishes the rows' outputs as well)
    launch_pairs(a, 1, st);
}

// ---- work items of 3..32 rows on the int8 matrix cores (q4k_mma_moe.hpp) ---------------------------------------------
// A dense Q4_K FFN (one expert, top-1, assignment i = row i) with at least 3 rows, in chunks of the sweep's width.
inline bool mma_dense(const mi355_moe_weights& w, const RowsK& r, uint32_t rows) {
    return w.gate_type == MI355_TYPE_Q4_K && w.down_type == MI355_TYPE_Q4_K && w.experts == 1U && w.top_k == 1U && rows >= 3U && !r.assignments;
}
// A decode batch whose expert's gate + up rows are several MB: one expert is swept once for the rows that chose it.
inline bool quad_sweep(const mi355_moe_weights& w, uint32_t rows);
inline bool large_expert(const mi355_moe_weights& w) { return 2ULL * w.ffn * (w.hidden / 256U) * kQ4kBlock >= (4ULL << 20); }
// Routed experts past the decode sizes or of several MB: the plan cuts an expert's rows into items of this
// many for the matrix-core sweeps (0: the vector-ALU sweeps serve the batch). The sweeps are bound by latency, so the narrow instances
// (4 or 8 rows: 123 or 142 registers, four or three waves per SIMD) win while an expert holds few rows, and even one row per expert is
// better off here than on the vector-ALU sweep. Layer times, hidden 2048 / ffn 768 / 128 experts top-8, items of 4 rows | of 16 in sweeps of 8 |
// in sweeps of 16 (vector-ALU sweep, which served up to 4 rows per expert): 17 rows 88 | - | 130 us (109), 28 rows 101 | 114 | 152 (126), 40
// rows 118 | 126 | 167 (147), 60 rows 141 | 139 | 181 (171), 100 rows 177 | 163 | 189, 200 rows 266 | 220 | 218, 400 rows 445 | 340 | 337; hidden
// 4096 / ffn 1536 / 64 experts: 24 rows 200 | 204 | 282 (260), 60 rows 300 | 267 | 288, 150 rows 550 | 439 | 414. A decode batch over large
// experts keeps its items of two rows: one rank's half of hidden 6144 / ffn 2560 / 160 experts, 7, 10, 16 rows: 189, 231, 306 us against 199,
// 251, 320; 10 rows of hidden 4096 / ffn 1536 / 64 experts, Q6_K | Q8_0 | Q5_K and Q5_1 rows: 271 | 271 | 258 -> 221 | 222 | 224 us.
// The other formats' batches, on their vector-ALU sweeps (items of four) before: hidden 2048 / ffn 768 / 128 experts, Q6_K down, 40, 300, 1000 rows
// 130, 395, 1105 -> 122, 258, 600 us; Q8_0 down 148, 440, 1203 -> 124, 245, 560; Q5_K gate / up and Q5_1 down 196, 774, 2310 -> 127, 264, 619.
// Items of up to four 32-row sweeps: the later sweeps of a tile's weights hit the cache, and an expert with thousands of rows
// still spreads over many workgroups.
constexpr uint32_t kMmaItemRows = 128;
inline bool q4k_both(const mi355_moe_weights& w) { return w.gate_type == MI355_TYPE_Q4_K && w.down_type == MI355_TYPE_Q4_K; }
// down rows of whole stages of 256 weights (Q8_0 and Q5_1 rows may end on half a stage)
inline bool mma_down_rows(const mi355_moe_weights& w) { return w.ffn % 256U == 0 && w.down_type != MI355_TYPE_Q5_K; }
// factors and sums that the sweeps' copies of 16 bytes take (a dense bundle is admitted with any of four; the vector-ALU sweeps, which read them
// word by word, serve items of any length)
inline bool mma_image(const A8Image& img) {
    return !img.table && aligned(img.deltas, 16) && aligned(img.sums, 16) && img.deltas_rs % 16U == 0 && img.sums_rs % 16U == 0;
}
inline uint32_t mma_grouped_split(const mi355_moe_weights& w, uint32_t rows) {
    if ((w.gate_type != MI355_TYPE_Q4_K && w.gate_type != MI355_TYPE_Q5_K) || w.experts == 1U) return 0U;
    if (rows <= kFusedMaxRows) return !quad_sweep(w, rows) && large_expert(w) ? 2U : 0U;
    const uint64_t assignments = static_cast<uint64_t>(rows) * w.top_k;
    if (!mma_down_rows(w) || assignments < 4ULL * w.experts) return 4U;
    return assignments < 16ULL * w.experts ? 16U : kMmaItemRows;
}
// rows of one sweep over such an item
inline uint32_t mma_sweep_rows(const mi355_moe_weights& w, uint32_t rows, uint32_t split) {
    return split == 16U && static_cast<uint64_t>(rows) * w.top_k < 12ULL * w.experts ? 8U : split;
}
// A dense FFN's gate and up rows as raw values into the intermediates, then the SwiGLU / A8 kernel (5..16 rows, one chunk).
inline void launch_mma_gate_up(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, hipStream_t st) {
    launch_mma_gate_up_rows(w, r, rows, st);
    swiglu_quantize_kernel<<<dim3((w.ffn / 32U + 7U) / 8U, rows), 256, 0, st>>>(r.gate_out, r.up_out, w.ffn, w.exp_kind, w.swiglu_limit, r.down_codes, r.down_deltas,
                                                                                r.down_sums, r.h_out, r.status, r.job_status);
}

inline void launch_plan(const PlanArgs& p, hipStream_t st) {
    if (p.assignments <= kPlanSmall) plan_small_kernel<<<1, 1024, 0, st>>>(p);
    else plan_kernel<<<p.experts, 1024, 0, st>>>(p);
}
// Decode batches of at most this many assignments (six tokens at top-8) run the 16-rows-per-wavefront sweep (q4k_quads.hpp),
// with a 4-slot ring up to 16 assignments and a 2-slot ring above (every workgroup of the launch stays resident); measured
// at hidden 2048 / ffn 768: faster than the 64-row sweep up to 48 assignments, slower at 64. Such a batch is planned one
// assignment per item (the fused router's plan, and the staged plan with pieces of one).
constexpr uint32_t kQuadMaxItems = 48;
inline bool quad_sweep(const mi355_moe_weights& w, uint32_t rows) {
    return rows <= kFusedMaxRows && rows * w.top_k <= kQuadMaxItems && w.experts > 1U;
}
// grouped: the fused router's plan of a decode batch with always-on experts, whose items hold up to four assignments; the narrow matrix-core
// sweeps serve it whatever its size (hidden 2048 / ffn 768 / 128 experts top-8 and one more, 5 rows, Q6_K | Q8_0 | Q4_K down: 88 | 93 | 86 -> 70 |
// 71 | 65 us; 1 row 53 | 54 | 52 -> 50 | 50 | 49; Q5_K gate / up and Q5_1 down without the norm 1, 2, 5, 16 rows 42.2, 54.0, 75.1, 132.7 -> 41.5,
// 46.8, 64.2, 115.2).
inline void launch_project(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t umax, hipStream_t st, bool grouped = false) {
    if (const uint32_t split = mma_grouped_split(w, rows); r.plan && mma_image(r.in) && (grouped || split))
        return launch_mma_project(w, r, rows, 0, umax, grouped ? 4U : mma_sweep_rows(w, rows, split), st);
    if (w.gate_type == MI355_TYPE_Q5_K) {
        // the deepest ring at which every workgroup of the launch is resident (4 waves x DEPTH x 4 KB each)
        const uint64_t groups = static_cast<uint64_t>(w.ffn / 32U) * umax;
        if (groups * 4U <= resident_waves(4U * kQuadSlotBytes)) project_q5k_kernel<4><<<dim3(w.ffn / 32U, umax), 256, 0, st>>>(w, r, rows * w.top_k);
        else project_q5k_kernel<2><<<dim3(w.ffn / 32U, umax), 256, 0, st>>>(w, r, rows * w.top_k);
        return;
    }
    if (!grouped && quad_sweep(w, rows)) {
        const uint32_t items = rows * w.top_k;
        if (items <= 16U) project_quad_kernel<4><<<dim3(w.ffn / 32U, items), 256, 0, st>>>(w, r, items);
        else project_quad_kernel<2><<<dim3(w.ffn / 32U, items), 256, 0, st>>>(w, r, items);
        return;
    }
    if (mma_dense(w, r, rows)) {
        if (rows > 4U && rows <= 16U && r.gate_out && r.up_out && dense_rows(r, w)) return launch_mma_gate_up(w, r, rows, st);
        return launch_mma_project(w, r, rows, rows, 0, rows, st);
    }
    if (dense_pairs_ok(w, rows) && dense_rows(r, w) && r.gate_out && r.up_out) return launch_project_dense(w, r, rows, st);
    const dim3 grid(w.ffn / 32U, umax);
    if (w.experts == 1U && rows > 4U) launch_project_nb<8>(w, r, rows, grid, st);
    else launch_project_nb<4>(w, r, rows, grid, st);
}
// Returns true when the launch also published the output rows (a dense top-1 job with r.top1_form set: the two dense sweeps).
inline bool launch_down(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t umax, hipStream_t st, bool grouped = false) {
    if (const uint32_t split = mma_grouped_split(w, rows); r.plan && mma_down_rows(w) && mma_image(r.h) && (grouped || split)) {
        RowsK plain = r;
        plain.top1_form = 0;
        launch_mma_down(w, plain, rows, 0, umax, grouped ? 4U : mma_sweep_rows(w, rows, split), st);
        return false;
    }
    if (w.down_type != MI355_TYPE_Q4_K) {      // Q8_0 / Q5_1 (blocks of 32, four chains per row) and Q6_K (pairs per super-block)
        const uint32_t assignments = rows * w.top_k, items_at = plan_items_at(w.experts, assignments), order_at = plan_order_at(w.experts);
        const dim3 grid(w.hidden / kDownGroupsRows, umax);
        // Q5_1 rows of whole super-blocks at 16-byte aligned addresses stream through a copy ring (its depth by residency)
        if (w.down_type == MI355_TYPE_Q5_1 && w.ffn % 256U == 0 && w.down_row_stride % 16U == 0 && w.down_expert_stride % 16U == 0 && mma_image(r.h)) {
            if (static_cast<uint64_t>(grid.x) * grid.y * 4U <= resident_waves(4U * group_slot_bytes())) down_q51_ring_kernel<4><<<grid, 256, 0, st>>>(w, r, assignments, items_at, order_at);
            else down_q51_ring_kernel<2><<<grid, 256, 0, st>>>(w, r, assignments, items_at, order_at);
        }
        else if (w.down_type == MI355_TYPE_Q8_0) down_groups_kernel<0><<<grid, 256, 0, st>>>(w, r, assignments, items_at, order_at);
        else if (w.down_type == MI355_TYPE_Q5_1) down_groups_kernel<1><<<grid, 256, 0, st>>>(w, r, assignments, items_at, order_at);
        else launch_down_q6k(w, r, grid, assignments, items_at, order_at, st);
        return false;
    }
    if (!grouped && quad_sweep(w, rows)) {
        const uint32_t items = rows * w.top_k;
        if (items <= 16U) down_quad_kernel<4><<<dim3(w.hidden / 64U, items), 256, 0, st>>>(w, r, items);
        else down_quad_kernel<2><<<dim3(w.hidden / 64U, items), 256, 0, st>>>(w, r, items);
        return false;
    }
    if (mma_dense(w, r, rows)) { launch_mma_down(w, r, rows, rows, 0, rows, st); return r.top1_form != 0; }
    if (dense_pairs_ok(w, rows) && dense_rows(r, w)) { launch_down_dense(w, r, rows, st); return r.top1_form != 0; }
    const dim3 grid(w.hidden / 64U, umax);
    if (w.experts == 1U && rows > 4U) launch_down_nb<8>(w, r, rows, grid, st);
    else launch_down_nb<4>(w, r, rows, grid, st);
    return false;
}
// An expert's assignments are cut into work items of at most `split` rows: a wave's instruction stream grows with every
// activation row it serves while its weight stream does not, so wide items finish last; the second read of a split
// expert's weights comes from the last-level cache. A dense matrix: every row shares one sweep.
inline uint32_t plan_split(const mi355_moe_weights& w, uint32_t rows) {
    if (w.experts == 1U) return 8;
    // decode batches on the vector-ALU sweeps: one item per assignment (the second sweep of an expert that two rows chose is a cache hit
    // while its gate + up rows are a few MB, and the short instruction streams finish sooner)
    const uint32_t split = mma_grouped_split(w, rows);
    return split ? split : 1U;
}
inline uint32_t item_bound(const mi355_moe_weights& w, uint32_t rows) {
    return plan_item_bound(w.experts, rows * w.top_k, plan_split(w, rows));
}
// Items by which a batch is admitted: of other formats than Q4_K those of four rows, however wide the batch's own are.
inline uint32_t admitted_items(const mi355_moe_weights& w, uint32_t rows) {
    const uint32_t split = plan_split(w, rows);
    return plan_item_bound(w.experts, rows * w.top_k, w.experts == 1U || q4k_both(w) || split < 4U ? split : 4U);
}

// ======================================================================================================== admission
// bytes of a GGUF row of k weights (k a multiple of 256)
inline uint64_t moe_row_bytes(uint32_t type, uint32_t k) {
    if (type == MI355_TYPE_Q8_0) return static_cast<uint64_t>(k / 32U) * kQ80Block;
    if (type == MI355_TYPE_Q5_1) return static_cast<uint64_t>(k / 32U) * 24U;
    if (type == MI355_TYPE_Q5_K) return static_cast<uint64_t>(k / 256U) * kQ5kBlock;
    if (type == MI355_TYPE_Q6_K) return static_cast<uint64_t>(k / 256U) * kQ6kBlock;
    return static_cast<uint64_t>(k / 256U) * kQ4kBlock;
}

// Tensor formats by arithmetic class. Integer-dot entries: gate/up Q4_K or Q5_K; down Q4_K, the host executor's Q8_0 /
// Q5_1 (src/cpu/core/routed_expert.hpp:27-28) or Q6_K (src/moe_a8_down_contract.cpp:147). The matrix-core prefill form: Q4_K, Q5_K or Q8_0 for either (a dense shared
// expert is experts = top_k = 1). The merge reads no weights.
enum MoeClass { kIntegerClass, kPrefillClass, kAnyClass };
int32_t check_moe(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, mi355_moe_weights& wv, MoeClass cls = kIntegerClass,
                  bool need_tensors = true) {
    STRIX_REQUIRE(w && r, "moe: null weights or rows");
    STRIX_REQUIRE(rows > 0, "moe: rows must be positive");
    const bool gate_q8 = w->gate_type == MI355_TYPE_Q8_0, down_q8 = w->down_type == MI355_TYPE_Q8_0;
    const bool down_q51 = w->down_type == MI355_TYPE_Q5_1 || w->down_type == MI355_TYPE_Q6_K;      // integer class only
    STRIX_REQUIRE(w->gate_type == MI355_TYPE_Q4_K || w->gate_type == MI355_TYPE_Q5_K || (gate_q8 && cls != kIntegerClass),
                  cls == kPrefillClass ? "moe prefill: gate/up weights must be Q4_K (type 12), Q5_K (type 13) or Q8_0 (type 8)" : "moe: gate/up weights must be Q4_K (type 12) or Q5_K (type 13)");
    if (!(w->down_type == MI355_TYPE_Q4_K || down_q8 || (down_q51 && cls != kPrefillClass) || (w->down_type == MI355_TYPE_Q5_K && cls != kIntegerClass)))
        return fail(MI355_E_UNSUPPORTED, cls == kPrefillClass ? "moe prefill: down weights must be Q4_K (type 12), Q5_K (type 13) or Q8_0 (type 8)"
                                                               : "moe: down weights must be Q4_K (type 12), Q8_0 (type 8), Q5_1 (type 7) or Q6_K (type 14)");
    STRIX_REQUIRE(w->hidden >= 256 && w->hidden % 256U == 0, "moe: hidden must be a positive multiple of 256");
    // K-quant down rows are super-blocks of 256; the executor's block-of-32 formats need four chains of groups (src/cpu/core/routed_expert.hpp:22)
    const uint32_t ffn_unit = (cls != kPrefillClass && (down_q8 || w->down_type == MI355_TYPE_Q5_1)) ? 128U : 256U;
    STRIX_REQUIRE(w->ffn >= ffn_unit && w->ffn % ffn_unit == 0, "moe: ffn must be a positive multiple of 256 (Q8_0 / Q5_1 down rows: 128)");
    STRIX_REQUIRE(w->experts > 0 && w->experts <= kRouteMaxExperts, "moe: experts must be within 1..1024");
    STRIX_REQUIRE(w->top_k > 0 && w->top_k <= kRouteMaxTopK && w->top_k <= w->experts, "moe: top_k must be within 1..16 and <= experts");
    STRIX_REQUIRE(static_cast<uint64_t>(rows) * w->top_k < (1ULL << 31), "moe: too many assignments");
    // rows are one grid dimension of the prologue and of the merge: every entry refuses a larger batch before its first launch
    STRIX_REQUIRE(rows <= 65535U, "moe: at most 65535 rows per call");
    // plan items are one grid dimension of the expert launches
    STRIX_REQUIRE(cls != kIntegerClass || admitted_items(*w, rows) <= 65535U, "moe: too many work items for one call (experts + rows * top_k / 4 must stay below 65536)");
    wv = *w;
    if (wv.gate_row_stride == 0) wv.gate_row_stride = moe_row_bytes(w->gate_type, w->hidden);
    if (wv.gate_expert_stride == 0) wv.gate_expert_stride = wv.gate_row_stride * w->ffn;
    if (wv.down_row_stride == 0) wv.down_row_stride = moe_row_bytes(w->down_type, w->ffn);
    if (wv.down_expert_stride == 0) wv.down_expert_stride = wv.down_row_stride * w->hidden;
    const uint32_t down_unit = w->down_type == MI355_TYPE_Q6_K ? 2U : 16U;        // Q6_K blocks are 210 bytes
    STRIX_REQUIRE(wv.gate_row_stride % 16U == 0 && wv.gate_expert_stride % 16U == 0 && wv.down_row_stride % down_unit == 0 &&
                  wv.down_expert_stride % down_unit == 0, "moe: weight strides must be multiples of 16 bytes (Q6_K down: 2)");
    STRIX_REQUIRE(wv.gate_row_stride < (1ULL << 27) && wv.down_row_stride < (1ULL << 27), "moe: weight row stride must be below 128 MiB");
    STRIX_REQUIRE(wv.gate_row_stride >= moe_row_bytes(w->gate_type, w->hidden) &&
                  wv.down_row_stride >= moe_row_bytes(w->down_type, w->ffn), "moe: weight row stride shorter than the row");
    // (a stage that reads no weights is admitted on the geometry alone)
    STRIX_REQUIRE(!need_tensors || (w->gate && w->up && w->down && aligned(w->gate, 16) && aligned(w->up, 16) && aligned(w->down, 16)),
                  "moe: weight pointers must be non-null and 16-byte aligned");
    STRIX_REQUIRE(w->exp_kind <= MI355_EXP_DECLARED, "moe: unknown exp kind");
    // the clamp trait: +infinity (or the zero-initialised 0) = none, else finite and positive (src/moe_a8_down_contract.cpp:57)
    if (wv.swiglu_limit == 0.0F) wv.swiglu_limit = INFINITY;
    STRIX_REQUIRE(wv.swiglu_limit > 0.0F, "moe: swiglu_limit must be +infinity (none) or finite and positive");
    STRIX_REQUIRE(r->routes && r->route_weights && r->codes && r->deltas && r->sums && r->status && r->down_codes && r->down_deltas &&
                  r->down_sums && r->rawdots && r->output && r->plan && r->job_status, "moe: a required row view is null");
    STRIX_REQUIRE(aligned(r->codes, 16) && aligned(r->down_codes, 16) && aligned(r->plan, 16) && aligned(r->rawdots, 16) &&
                  aligned(r->deltas, 4) && aligned(r->down_deltas, 4), "moe: row views must be 16-byte aligned");
    STRIX_REQUIRE(r->output_stride >= w->hidden, "moe: output stride shorter than hidden");
    return MI355_OK;
}

}  // namespace strix950

// ============================================================================================================ C ABI
using namespace strix950;

extern "C" {

const char* mi355_last_error(void) { return g_error.c_str(); }
const char* mi355_version(void) { return "mi355-strix 0.1 (gfx950)"; }

const char* mi355_numerical_identity(uint32_t weight_type, int down) {
    // Identity strings are the admission tokens of the reference's contracts (include/strix/moe_q4k_a8_contract.hpp:24-29,
    // include/strix/moe_a8_down_contract.hpp:9-28); a caller hands over the token of the arithmetic it approved. The tokens are
    // returned verbatim because the bits are the same: "wave32" in the probe tokens names the reference's reduction tree
    // (pairs ascending, four super-block partials folded by a two-level tree), which the 64-lane kernels here reproduce.
    if (!down) {
        if (weight_type == MI355_TYPE_Q4_K)
            return "strix-moe-q4k-a8g32-probe-v2:f32-div-rne:g32-sym127-zero1-finite-noflush:"
                   "dot-s8xu8-i32:combine-separate-f32:pair-ascending-sb-tree4:writer-c0:wave32:proj-nonfinite=propagate-unqualified";
        if (weight_type == MI355_TYPE_Q5_K)
            return "strix-moe-q5k-a8g32-probe-v1:f32-div-rne:g32-sym127-zero1-finite-noflush:"
                   "dot-s8xu5qh-i32:combine-separate-f32:pair-ascending-sb-tree4:writer-c0:wave32:proj-nonfinite=propagate-unqualified";
        if (weight_type == MI355_TYPE_Q8_0) return "cpu-q8a8-tree32@1";
        return "";
    }
    if (weight_type == MI355_TYPE_Q4_K)
        return "q4k-a8g32-down-v1:s8xu4-i32:delta*((d*(sc*I))-(dmin*(m*S))):pair-ascending-sb-tree4:"
               "silu-div-expf-times-up:g32-sym127-f32delta-rne:tiny-lt2^-119-zero1:raw-slot-major:finite-failclosed";
    if (weight_type == MI355_TYPE_Q6_K)
        return "q6k-a8g32-down-v1:s8xs8-i32:delta*(d*(s0*I0+s1*I1)):pair-ascending-sb-tree4:"
               "silu-div-expf-times-up:g32-sym127-f32delta-rne:tiny-lt2^-119-zero1:raw-slot-major:finite-failclosed";
    if (weight_type == MI355_TYPE_Q5_1)
        return "q51-a8g32-down-v1:s8xu5-i32:delta*(d*S+m*C):separate-f32:"
               "silu-div-expf-times-up:g32-sym127-f32delta-rne:tiny-lt2^-119-zero1:"
               "blocks-mod4-ascending:tree-xor1-xor2:raw-slot-major:finite-failclosed";
    if (weight_type == MI355_TYPE_Q8_0)
        return "q80-a8g32-down-v1:s8xs8-i32:delta*(d*S):separate-f32:"
               "silu-div-expf-times-up:g32-sym127-f32delta-rne:tiny-lt2^-119-zero1:"
               "blocks-mod4-ascending:tree-xor1-xor2:raw-slot-major:finite-failclosed";
    return "";
}

int32_t mi355_dequantize_rows(uint32_t type, const void* rows, uint64_t row_stride, uint32_t n_rows, uint32_t elements,
                              float* out, uint64_t out_stride, mi355_stream stream) {
    if (type != MI355_TYPE_Q8_0 && type != MI355_TYPE_Q4_K) return fail(MI355_E_UNSUPPORTED, "dequantize: type must be Q8_0 (8) or Q4_K (12)");
    const uint32_t be = type == MI355_TYPE_Q8_0 ? 32U : 256U, bb = type == MI355_TYPE_Q8_0 ? kQ80Block : kQ4kBlock;
    STRIX_REQUIRE(rows && out, "dequantize: null pointer");
    STRIX_REQUIRE(elements % be == 0, "dequantize: row length is not a multiple of the block");
    STRIX_REQUIRE(row_stride >= static_cast<uint64_t>(elements / be) * bb && out_stride >= elements, "dequantize: stride shorter than the row");
    if (n_rows == 0 || elements == 0) return MI355_OK;
    const uint32_t gx = (elements + 255U) / 256U;
    for (uint32_t r0 = 0; r0 < n_rows; r0 += 65535U) {
        const uint32_t nr = n_rows - r0 < 65535U ? n_rows - r0 : 65535U;
        dequantize_rows_kernel<<<dim3(gx < 64U ? gx : 64U, nr), 256, 0, hs(stream)>>>(
            type, static_cast<const uint8_t*>(rows) + r0 * row_stride, row_stride, elements, out + r0 * out_stride, out_stride);
    }
    STRIX_LAUNCHED("dequantize_rows");
    return MI355_OK;
}

int32_t mi355_quantize_weight_rows(uint32_t type, const float* x, uint32_t n_rows, uint32_t elements, void* out, mi355_stream stream) {
    if (type != MI355_TYPE_Q8_0 && type != MI355_TYPE_Q4_K) return fail(MI355_E_UNSUPPORTED, "quantize_weight: type must be Q8_0 (8) or Q4_K (12)");
    const uint32_t be = type == MI355_TYPE_Q8_0 ? 32U : 256U;
    STRIX_REQUIRE(x && out, "quantize_weight: null pointer");
    STRIX_REQUIRE(elements % be == 0, "quantize_weight: row length is not a multiple of the block");
    const uint64_t blocks = static_cast<uint64_t>(n_rows) * (elements / be);
    if (blocks == 0) return MI355_OK;
    if (type == MI355_TYPE_Q8_0) {
        const uint64_t g = (blocks + 255U) / 256U;
        quantize_q8_0_rows_kernel<<<static_cast<uint32_t>(g < 65535U ? g : 65535U), 256, 0, hs(stream)>>>(x, blocks, static_cast<uint8_t*>(out));
    } else {
        const uint64_t g = (blocks + 63U) / 64U;
        quantize_q4_k_rows_kernel<<<static_cast<uint32_t>(g < 262144U ? g : 262144U), 64, 0, hs(stream)>>>(x, blocks, static_cast<uint8_t*>(out));
    }
    STRIX_LAUNCHED("quantize_weight_rows");
    return MI355_OK;
}

int32_t mi355_rmsnorm_f32(const float* x, const float* w, uint32_t n, float eps, float* y, uint32_t rows, mi355_stream stream) {
    if (rows == 0 || n == 0) return MI355_OK;
    STRIX_REQUIRE(x && y, "rmsnorm: null pointer");
    STRIX_REQUIRE(rows <= 0x7fffffffU, "rmsnorm: too many rows");
    rmsnorm_f32_kernel<<<rows, n >= 512U ? 256 : 128, 0, hs(stream)>>>(x, w, n, eps, y);
    STRIX_LAUNCHED("rmsnorm_f32");
    return MI355_OK;
}

namespace {
int32_t check_route(const mi355_route_policy* p, const void* x, uint32_t kind, uint32_t hidden, uint64_t x_stride, const float* wr,
                    const uint32_t* ids, const float* weights, const float* scores) {
    STRIX_REQUIRE(p && x && wr && ids && weights && scores, "route: null pointer");
    STRIX_REQUIRE(p->experts > 0 && p->experts <= kRouteMaxExperts && p->top_k > 0 && p->top_k <= kRouteMaxTopK && p->top_k <= p->experts,
                  "route policy: need 0 < top_k <= experts, experts <= 1024, top_k <= 16");
    STRIX_REQUIRE(p->shared_experts <= 4U && p->top_k + p->shared_experts <= kRouteMaxTopK && p->experts + p->shared_experts <= kRouteMaxExperts,
                  "route policy: at most 4 always-on experts, top_k + shared <= 16, experts + shared <= 1024");
    STRIX_REQUIRE(hidden > 0 && hidden <= kRouteMaxHidden && hidden % 32U == 0, "route: hidden must be a multiple of 32 within 16384");
    STRIX_REQUIRE(kind <= MI355_INPUT_BF16 && p->logits_order <= MI355_LOGITS_LANE32_BUTTERFLY, "route: unknown input kind or logits order");
    STRIX_REQUIRE(p->exp_kind <= MI355_EXP_LIBM, "route policy: unknown exp kind");
    STRIX_REQUIRE(aligned(wr, 16) && aligned(x, 16) && x_stride % 16U == 0, "route: router weight, activations and their row stride must be 16-byte aligned");
    return MI355_OK;
}
// Logits of every (row, expert) into a.scores. Decode batches: one block per (row, 8 experts), plus a.quant_blocks blocks
// in the fused form; larger batches: route.hip.
void launch_route_logits(RouteArgs& a, hipStream_t st) {
    const uint32_t neb = (a.p.experts + 7U) / 8U;
    // Logits alone of rows past 2048 features: on the matrix cores, whose chain is the faster one (8.9 cycles a feature against 10.1 of the vector ALU) and starts
    // later. Hidden 1024, 2048, 6144, 16 rows, vector ALU | matrix cores, with the selection, 9.8, 14.6, 32.1 | 10.2, 14.4, 29.6 us (fp32 rows of 6144 34.2 | 29.5).
    const bool alone = !a.quant_blocks && a.p.logits_order == MI355_LOGITS_FMA_ASCENDING && a.hidden > 2048U;
    if (a.rows <= kFusedMaxRows && !alone) {
        a.route_blocks = neb * a.rows;
        const uint32_t blocks = a.route_blocks + a.quant_blocks;
        const auto launch = [&](auto norm) {
            constexpr bool NORM = decltype(norm)::value;
            if (a.kind == MI355_INPUT_F32) route_decode_kernel<0, NORM><<<blocks, 64, 0, st>>>(a);
            else if (a.kind == MI355_INPUT_F16) route_decode_kernel<1, NORM><<<blocks, 64, 0, st>>>(a);
            else route_decode_kernel<2, NORM><<<blocks, 64, 0, st>>>(a);
        };
        if (a.normed) launch(std::true_type{});
        else launch(std::false_type{});
    } else launch_route_batch_logits(a, st);
}
}  // namespace

int32_t mi355_moe_route(const mi355_route_policy* p, const void* x, uint32_t kind, uint32_t rows, uint32_t hidden, uint64_t x_stride,
                        const float* wr, const float* bias, uint32_t* ids, float* weights, float* scores, mi355_stream stream) {
    if (const int32_t rc = check_route(p, x, kind, hidden, x_stride, wr, ids, weights, scores)) return rc;
    if (rows == 0) return MI355_OK;
    RouteArgs a{};
    a.p = *p; a.x = static_cast<const uint8_t*>(x); a.kind = kind; a.x_stride = x_stride; a.rows = rows; a.hidden = hidden;
    a.wr = wr; a.bias = bias; a.ids = ids; a.weights = weights; a.scores = scores;
    launch_route_logits(a, hs(stream));
    launch_route_select(a, hs(stream));
    STRIX_LAUNCHED("moe_route");
    return MI355_OK;
}

size_t mi355_moe_prefill_f16_workspace_bytes(uint32_t hidden, uint32_t ffn, uint32_t rows, uint32_t top_k) {
    return pf_workspace_bytes(hidden, ffn, rows, top_k);
}

size_t mi355_moe_plan_words(uint32_t experts, uint32_t rows, uint32_t top_k) {
    return plan_words_total(experts, rows * top_k);
}

}  // extern "C"
namespace {
RouteCheck route_check(const mi355_moe_weights& wv, const mi355_moe_rows& r) {
    return RouteCheck{r.routes, r.route_weights, wv.experts, wv.top_k, r.status, r.job_status};
}
PlanArgs batch_plan(const mi355_moe_weights& wv, const mi355_moe_rows& r, uint32_t rows) {
    return PlanArgs{dense_routes(r.routes, wv.top_k), wv.experts, rows * wv.top_k, plan_split(wv, rows), item_bound(wv, rows), r.plan};
}
// plan: the batch's plan as well
int32_t enqueue_prologue_rows(const mi355_moe_weights& wv, const mi355_moe_rows& r, uint32_t rows, bool plan, hipStream_t st) {
    STRIX_REQUIRE(r.codes && r.deltas, "A8: null pointer");
    STRIX_REQUIRE(rows <= 65535U, "A8: at most 65535 rows per call");
    const bool vec = aligned(r.input, 16) && r.input_stride % 16U == 0 && aligned(r.codes, 8);
    launch_prologue_rows(A8RowArgs{static_cast<const uint8_t*>(r.input), r.input_stride, wv.hidden, r.codes, r.deltas, r.sums, nullptr, kA8StatusNone, vec, 0U},
                         r.input_kind, rows, route_check(wv, r), plan ? batch_plan(wv, r, rows) : PlanArgs{}, st);
    STRIX_LAUNCHED("moe prologue");
    return MI355_OK;
}
}  // namespace
extern "C" {
int32_t mi355_moe_enqueue_prologue(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, mi355_stream stream) {
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv)) return rc;
    STRIX_REQUIRE(r->input && r->input_kind <= MI355_INPUT_BF16, "moe prologue: input view invalid");
    return enqueue_prologue_rows(wv, *r, rows, false, hs(stream));
}

int32_t mi355_moe_enqueue_csr(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, mi355_stream stream) {
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv)) return rc;
    launch_plan(batch_plan(wv, *r, rows), hs(stream));
    STRIX_LAUNCHED("moe plan");
    return MI355_OK;
}

int32_t mi355_moe_enqueue_project(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, mi355_stream stream) {
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv)) return rc;
    launch_project(wv, rows_k(*r, wv), rows, item_bound(wv, rows), hs(stream));
    STRIX_LAUNCHED("moe project");
    return MI355_OK;
}

int32_t mi355_moe_enqueue_down(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, mi355_stream stream) {
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv)) return rc;
    launch_down(wv, rows_k(*r, wv), rows, item_bound(wv, rows), hs(stream));
    STRIX_LAUNCHED("moe down");
    return MI355_OK;
}

}  // extern "C"
namespace {
// shared_slots: the last slots of every row are always-on experts (a layer call with policy->shared_experts)
int32_t enqueue_merge(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream, uint32_t shared_slots) {
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv, kAnyClass)) return rc;
    STRIX_REQUIRE(form <= MI355_COMBINE_MULADD_ASCENDING_EXPERT, "moe merge: unknown combine form");
    STRIX_REQUIRE(rows <= 65535U, "moe merge: at most 65535 rows per call");
    RowsK k = rows_k(*r, wv);
    k.shared_slots = shared_slots;
    // four columns per thread once that still leaves every compute unit two workgroups (333 rows x 2048, 666 workgroups: 6.9 -> 6.3 us;
    // a decode batch is faster with one column per thread: 16 rows x 6144: 5.0 against 6.1 us)
    const bool quads = static_cast<uint64_t>(rows) * ((wv.hidden + 1023U) / 1024U) >= 2ULL * compute_units() && wv.hidden % 4U == 0 && aligned(k.rawdots, 16) && k.rawdots_rs % 16U == 0 && aligned(k.output, 16) && k.output_stride % 4U == 0 &&
                       (!k.base || (aligned(k.base, 16) && k.base_rs % 16U == 0));
    if (quads) merge_kernel<4><<<dim3((wv.hidden + 1023U) / 1024U, rows), 256, 0, hs(stream)>>>(wv, k, form);
    else merge_kernel<1><<<dim3((wv.hidden + 255U) / 256U, rows), 256, 0, hs(stream)>>>(wv, k, form);
    STRIX_LAUNCHED("moe merge");
    return MI355_OK;
}
}  // namespace
extern "C" {

int32_t mi355_moe_enqueue_merge(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream) {
    return enqueue_merge(w, r, rows, form, stream, 0U);
}

int32_t mi355_moe_enqueue(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream) {
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv)) return rc;   // the whole bundle is validated before the first enqueue
    STRIX_REQUIRE(form <= MI355_COMBINE_MULADD_ASCENDING_EXPERT, "moe: unknown combine form");
    STRIX_REQUIRE(r->input && r->input_kind <= MI355_INPUT_BF16, "moe: input view invalid");
    // a dense matrix on the pair-per-lane sweep reads no expert plan
    if (const int32_t rc = enqueue_prologue_rows(wv, *r, rows, !(dense_pairs_ok(wv, rows) && r->gate_out && r->up_out), hs(stream))) return rc;
    if (const int32_t rc = mi355_moe_enqueue_project(w, r, rows, stream)) return rc;
    // a dense top-1 job: the down launch publishes each row's output with its one unweighted value (no merge launch)
    RowsK k = rows_k(*r, wv);
    if (wv.experts == 1U && wv.top_k == 1U && rows <= 65535U) k.top1_form = form + 1U;
    const bool published = launch_down(wv, k, rows, item_bound(wv, rows), hs(stream));
    STRIX_LAUNCHED("moe down");
    if (published) return MI355_OK;
    return mi355_moe_enqueue_merge(w, r, rows, form, stream);
}

}  // extern "C"

namespace {
// mi355_moe_enqueue by halves: front = prologue, plan, gate / up; back = down rows, combine.
int32_t enqueue_staged(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream, bool do_front, bool do_back,
                       uint32_t shared_slots = 0) {
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv)) return rc;
    STRIX_REQUIRE(form <= MI355_COMBINE_MULADD_ASCENDING_EXPERT, "moe: unknown combine form");
    if (do_front) {
        STRIX_REQUIRE(r->input && r->input_kind <= MI355_INPUT_BF16, "moe: input view invalid");
        if (const int32_t rc = enqueue_prologue_rows(wv, *r, rows, !(dense_pairs_ok(wv, rows) && r->gate_out && r->up_out), hs(stream))) return rc;
        if (const int32_t rc = mi355_moe_enqueue_project(w, r, rows, stream)) return rc;
    }
    if (!do_back) return MI355_OK;
    RowsK k = rows_k(*r, wv);
    if (wv.experts == 1U && wv.top_k == 1U && rows <= 65535U) k.top1_form = form + 1U;
    const bool published = launch_down(wv, k, rows, item_bound(wv, rows), hs(stream));
    STRIX_LAUNCHED("moe down");
    if (published) return MI355_OK;
    return enqueue_merge(w, r, rows, form, stream, shared_slots);
}

struct LayerNorm { bool on; const float* weight; float eps; float* normed; };
std::atomic<uint32_t> g_early_perturb{0};
std::atomic<bool> g_down_merge_flat{true};

// phase: 0 = the whole layer; 1 = its front half (router, A8 prologue, plan, gate / up); 2 = its back half (down rows, combine) on
// what a front call with the same arguments left in the row views.
enum { kLayerWhole = 0, kLayerFront = 1, kLayerBack = 2 };
// down rows + combine of a decode batch whose every workgroup is resident: dense rows of at most four super-blocks stream as
// contiguous stages (down_merge_flat_kernel), other shapes as 144-byte blocks of 64 rows (down_merge_kernel)
void launch_down_merge(const mi355_moe_weights& wv, const RowsK& k, uint32_t rows, uint32_t items, uint32_t form, hipStream_t st) {
    const dim3 grid(wv.hidden / 64U, rows);
    const uint32_t threads = 64U * wv.top_k, B = wv.ffn / 256U;
    const bool flat = wv.down_row_stride == static_cast<uint64_t>(B) * kQ4kBlock && wv.down_expert_stride % 16U == 0 && !k.h.table && k.h.codes &&
                      aligned(k.h.codes, 16) && aligned(k.h.deltas, 16) && aligned(k.h.sums, 16) && wv.ffn % 256U == 0 && g_down_merge_flat.load(std::memory_order_relaxed);
    if (flat && B == 1U) down_merge_flat_kernel<1><<<grid, threads, 0, st>>>(wv, k, items, form);
    else if (flat && B == 2U) down_merge_flat_kernel<2><<<grid, threads, 0, st>>>(wv, k, items, form);
    else if (flat && B == 3U) down_merge_flat_kernel<3><<<grid, threads, 0, st>>>(wv, k, items, form);
    else if (flat && B == 4U) down_merge_flat_kernel<4><<<grid, threads, 0, st>>>(wv, k, items, form);
    else down_merge_kernel<<<grid, threads, 0, st>>>(wv, k, items, form);
}
// launch(SLOTS): of the instance for that many slots. Nine, top-8 and an always-on expert, have one of their own: more workgroups a compute unit than with sixteen slots' LDS, more registers than
// waves of 1024 threads may have. Layers of 2048 / 768 / 128 with it, instance of sixteen | nine, 1, 5, 12 rows, us: Q4_K 31.9, 46.3, 76.0 | 31.4, 44.4, 71.7; Q6_K 30.1, 49.0, 84.8 | 29.9,
// 47.0, 81.1; Q8_0 29.9, 49.0, 83.7 | 30.0, 48.6, 82.6; Q5_1 30.1, 50.3, 84.6 | 29.8, 48.2, 79.6.
template <class Launch> void down_merge_slots(uint32_t slots, Launch launch) {
    if (slots <= kDownMergeSlots) launch(std::integral_constant<uint32_t, kDownMergeSlots>{});
    else if (slots == kDownMergeSlots + 1U) launch(std::integral_constant<uint32_t, kDownMergeSlots + 1U>{});
    else launch(std::integral_constant<uint32_t, kDownMergeMost>{});
}
// The other formats' down rows + combine, 16 output columns a workgroup: which launches they take, and the launch.
bool down_merge_format_takes(const mi355_moe_weights& wv, const A8Image& h, uint32_t rows) {
    if (wv.top_k > kDownMergeMost || wv.hidden % 16U != 0 || rows > 65535U) return false;
    if (wv.down_type == MI355_TYPE_Q8_0) return wv.ffn % 128U == 0;
    if (wv.down_type == MI355_TYPE_Q5_1) return wv.ffn % 256U == 0 && wv.down_row_stride % 16U == 0 && wv.down_expert_stride % 16U == 0 && mma_image(h);      // (what down_q51_ring_kernel's copies need)
    return wv.down_type == MI355_TYPE_Q6_K;
}
bool launch_down_merge_format(const mi355_moe_weights& wv, const RowsK& k, uint32_t rows, uint32_t items, uint32_t form, hipStream_t st) {
    if (!down_merge_format_takes(wv, k.h, rows)) return false;
    const dim3 grid(wv.hidden / 16U, rows);
    down_merge_slots(wv.top_k, [&](auto slots) {
        constexpr uint32_t SLOTS = decltype(slots)::value;
        if (wv.down_type == MI355_TYPE_Q8_0) down_merge_q8_0_kernel<SLOTS><<<grid, 64U * wv.top_k, 0, st>>>(wv, k, items, form);
        else if (wv.down_type == MI355_TYPE_Q5_1) down_merge_q51_kernel<2, SLOTS><<<grid, 64U * wv.top_k, 0, st>>>(wv, k, items, form);
        else down_merge_q6k_kernel<SLOTS><<<grid, 64U * wv.top_k, 0, st>>>(wv, k, items, form);
    });
    return true;
}
// Q4_K down rows, 16 columns a workgroup (rings of four slots for one or two rows, where eight of them fit)
void launch_down_merge_quad(const mi355_moe_weights& wv, const RowsK& k, uint32_t rows, uint32_t items, uint32_t form, hipStream_t st) {
    const dim3 grid(wv.hidden / kQuadRows, rows);
    down_merge_slots(wv.top_k, [&](auto slots) {
        constexpr uint32_t SLOTS = decltype(slots)::value;
        if (SLOTS == kDownMergeSlots && rows <= 2U) down_merge_quad_kernel<SLOTS == kDownMergeSlots ? 4 : 2, SLOTS><<<grid, 64U * wv.top_k, 0, st>>>(wv, k, items, form);
        else down_merge_quad_kernel<2, SLOTS><<<grid, 64U * wv.top_k, 0, st>>>(wv, k, items, form);
    });
}

int32_t enqueue_layer(const mi355_route_policy* p, const float* router_weight, const float* logit_bias, float* scores, const LayerNorm& norm,
                      const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream, uint32_t phase = kLayerWhole) {
    const bool do_front = phase != kLayerBack, do_back = phase != kLayerFront;
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv)) return rc;
    const auto layer_rows = [&] { RowsK k = rows_k(*r, wv); k.shared_slots = p->shared_experts; return k; };
    STRIX_REQUIRE(form <= MI355_COMBINE_MULADD_ASCENDING_EXPERT, "moe: unknown combine form");
    STRIX_REQUIRE(r->input && r->input_kind <= MI355_INPUT_BF16, "moe: input view invalid");
    uint32_t* ids = const_cast<uint32_t*>(r->routes);
    float* weights = const_cast<float*>(r->route_weights);
    if (const int32_t rc = check_route(p, r->input, r->input_kind, wv.hidden, r->input_stride, router_weight, ids, weights, scores)) return rc;
    STRIX_REQUIRE(p->experts + p->shared_experts == wv.experts && p->top_k + p->shared_experts == wv.top_k,
                  "moe layer: router policy (experts, top_k, always-on experts) and expert tensors disagree on experts / top_k");
    STRIX_REQUIRE(!norm.on || (norm.normed && aligned(norm.normed, 16) && (!norm.weight || aligned(norm.weight, 16)) && norm.eps >= 0.0F),
                  "moe layer: the RMSNorm needs a 16-byte aligned fp32 [rows][hidden] view for the normalised rows, aligned weights, eps >= 0");
    hipStream_t st = hs(stream);
    const auto norm_rows = [&] { launch_norm_rows(r->input, r->input_kind, r->input_stride, norm.weight, wv.hidden, norm.eps, norm.normed, rows, st); };
    if (rows > kFusedMaxRows || plan_split(wv, rows) != 1U) {      // large batches, and decode batches over large experts (shared sweeps): router, then the staged prologue / plan
        mi355_moe_rows staged = *r;
        if (norm.on && do_front) {
            norm_rows();
            STRIX_LAUNCHED("moe layer norm");
        }
        if (norm.on) { staged.input = norm.normed; staged.input_kind = MI355_INPUT_F32; staged.input_stride = 4ULL * wv.hidden; }
        RouteArgs a{};
        a.p = *p; a.x = static_cast<const uint8_t*>(staged.input); a.kind = staged.input_kind; a.x_stride = staged.input_stride; a.rows = rows; a.hidden = wv.hidden;
        a.wr = router_weight; a.bias = logit_bias; a.ids = ids; a.weights = weights; a.scores = scores;
        if (do_front) {
            if (const int32_t rc = check_route(p, staged.input, staged.input_kind, wv.hidden, staged.input_stride, router_weight, ids, weights, scores)) return rc;
            launch_route_logits(a, st);
            launch_route_select(a, st);
            STRIX_LAUNCHED("moe layer router");
        }
        return enqueue_staged(w, &staged, rows, form, stream, do_front, do_back, p->shared_experts);
    }
    RouteArgs a{};
    a.p = *p; a.x = static_cast<const uint8_t*>(r->input); a.kind = r->input_kind; a.x_stride = r->input_stride; a.rows = rows; a.hidden = wv.hidden;
    a.wr = router_weight; a.bias = logit_bias; a.ids = ids; a.weights = weights; a.scores = scores;
    a.codes = r->codes; a.deltas = r->deltas; a.sums = r->sums; a.status = r->status; a.job_status = r->job_status; a.plan = r->plan;
    a.quant_blocks = (rows * (wv.hidden / 32U) + 7U) / 8U;
    const uint32_t items = rows * wv.top_k;
    // Early routes (route_early.hpp): the expert choice from lane-parallel logits in a short first launch, the exact router beside
    // the projection, down rows + combine on the verified work items. Taken where the 64-row projection sweep and the down +
    // combine launch serve the batch.
    // From 8 assignments on (one row of top-8): measured at hidden 2048 / ffn 768 against the three launches of the smallest batches
    // (router, 16-row projection, 16-row down + combine): 1 row 28.7 / 31.3 us, 2 rows 31.6 / 35.4, 3 rows 33.4 / 37.8, 4 rows
    // 35.7 / 40.3, 5 rows 38.4 / 48.6, 6 rows 41.2 / 57.8.
    // Down rows of another format, 1, 8, 16 rows against the router launch, the projection and the same down + combine launch: Q6_K 31.6, 67.5,
    // 111.8 -> 26.2, 58.5, 95.2 us, Q8_0 31.0, 67.6, 111.7 -> 25.3, 58.6, 92.1, Q5_1 30.8, 61.0, 100.5 -> 24.9, 52.0, 83.8.
    // Any width, however many rounds the down + combine launch's workgroups take (each of 64 columns fills a compute unit's LDS). Router launch, projection,
    // down rows -> early routes, rows of hidden / ffn / experts, top-8: 1 of 2304 / 768 / 64 32.9 -> 30.4 us, 1 of 4096 / 1536 / 64 51.4 -> 48.5, 1 of 6144 / 2560 / 160
    // 107.2 -> 79.3, 4 of 4096 / 1536 / 64 101.5 -> 77.3, 8 of 4096 / 768 / 128 93.9 -> 75.9, 16 of them 156.5 -> 127.2, 16 of 5120 / 512 / 128 143.6 -> 123.4; fp32 rows, 5 of 6144 / 768 / 64
    // 103.2 -> 79.9; Q8_0 down rows, 16 of 4096 / 768 / 128 192.4 -> 164.4; top-16 and top-10, 1, 4 rows of 2048 / 768 / 128 36.8, 49.8 -> 29.7, 39.5. Batches of more than
    // kQuadMaxItems assignments over large experts share their sweeps instead (above): 16 rows of one rank's half of 6144 / 2560 / 160 291.6, with early routes 352.1.
    // Always-on experts: a row's slot more, whose weights every row sweeps by itself where the plan of the router launch has four rows share a sweep. 1, 2, 5, 8, 14
    // rows of 2048 / 768 / 128 40.4, 43.7, 59.1, 72.4, 94.7 -> 31.8, 32.3, 48.3, 61.7, 88.0 us, Q6_K down rows 41.8, 45.9, 62.4, 79.2, 106.5 -> 32.5, 34.2, 55.4, 71.7, 104.1, 4 rows of
    // 4096 / 1536 / 64 111.4 -> 91.8. What the shared sweeps save grows with the bytes of these weights over the rows, what the early routes save with the chain: the line lies at 32 KiB a
    // feature, up to 3072 features at no more than 64 MiB. Router launch | early routes (MiB of them), us: 2048 / 2560 top-4, 7, 9 rows (59, 76) 81.7 | 75.7, 93.5 | 97.6; 1792 / 2048
    // top-4, 9, 10 (53, 59) 78.7 | 77.7, 82.1 | 92.4; 3072 / 2048 top-4, 6, 7, 8 (61, 71, 81) 89.5 | 87.4, 96.3 | 101.2, 103.3 | 105.1; 3840 / 2048 top-4, 7, 9 (89, 114) 117.0 | 113.6,
    // 135.3 | 135.9; 5120 / 2048 top-4, 6, 8 (101, 135) 135.0 | 114.6, 157.4 | 153.6; 6144 / 2560, 3 rows top-8 (76) 176.8 | 172.4, 8 top-2 (202) 139.3 | 130.1. Rows of up to
    // kChainNormHidden features, whose chain is short and which the router launch norms for nothing, only of experts no wider than they are long and five slots: 8 rows of 1280 / 2048
    // top-4 63.0 | 65.5, 7 of 1024 / 2560 top-2 42.6 | 45.8, 8 of 1536 / 1536 top-4 56.4 | 51.6, 1, 4, 14 of 1024 / 512 / 128 37.6, 37.4, 55.3 | 31.2, 31.1, 42.1, with the norm 38.6, 38.2, 58.1 |
    // 33.8, 33.2, 44.4, 14 of 1280 / 1024 / 64 with the norm, Q6_K, Q8_0 down rows 93.9, 92.0 | 88.2, 89.3, 6 of 1280 / 768 top-4 with it 41.0 | 35.1. (Three slots with it gain no more
    // than runs of one program differ, 16 rows of 1024 / 512 37.0 | 35.1, without it 37.9 | 30.9.)
    const RowsK k = [&] { RowsK view = layer_rows(); view.awords = r->plan + kPlanAwordsAt; return view; }();
    const uint64_t expert_bytes = 2ULL * wv.ffn * moe_row_bytes(wv.gate_type, wv.hidden) + static_cast<uint64_t>(wv.hidden) * moe_row_bytes(wv.down_type, wv.ffn);
    const uint64_t most = wv.hidden > 2048U && wv.hidden <= 3072U ? 64ULL << 20 : static_cast<uint64_t>(wv.hidden) << 15;
    const bool always_on = p->shared_experts == 0 || ((wv.hidden > kChainNormHidden || (wv.ffn <= wv.hidden && wv.top_k >= 5U)) && p->shared_experts * rows * expert_bytes <= most);
    const bool early = always_on && p->logits_order == MI355_LOGITS_FMA_ASCENDING && wv.gate_type == MI355_TYPE_Q4_K &&
                       (wv.down_type == MI355_TYPE_Q4_K || down_merge_format_takes(wv, k.h, rows)) && items >= kEarlyMinAssignments && wv.experts > 1U && wv.top_k <= kDownMergeMost &&
                       items <= kEarlyMaxAssignments && wv.hidden % 64U == 0 && 2U * wv.experts <= wv.top_k * wv.hidden;
    // (rows that are normalised in place: the router's workgroups would read what others of their launch have written)
    const uint64_t raw = reinterpret_cast<uint64_t>(r->input), raw_end = raw + (rows - 1U) * r->input_stride + (r->input_kind == MI355_INPUT_F32 ? 4ULL : 2ULL) * wv.hidden;
    const uint64_t out = reinterpret_cast<uint64_t>(norm.normed), out_end = out + 4ULL * rows * wv.hidden;
    const bool in_place = raw < out_end && out < raw_end;
    if (norm.on && (early || wv.hidden > kChainNormHidden || in_place)) {
        // The normalised rows in a launch of their own; the router takes them as fp32 rows. (In the router's launch every workgroup works its
        // row's factor out again, in front of its chain. Layers of 1 row x 4096, 3 x 6144, 8 x 3072, 16 x 4096 fp32 rows: 60.5, 86.5, 74.5,
        // 139.4 us, with this launch 46.6, 62.1, 67.3, 96.8; 5 rows of 2048 with an always-on expert 64.2 -> 61.0.)
        if (do_front) norm_rows();
        a.x = reinterpret_cast<const uint8_t*>(norm.normed); a.kind = MI355_INPUT_F32; a.x_stride = 4ULL * wv.hidden;
    } else if (norm.on) { a.norm_w = norm.weight; a.norm_eps = norm.eps; a.normed = norm.normed; }
    if (early) {
        a.awords = r->plan + kPlanAwordsAt;
        a.early_perturb = g_early_perturb.load(std::memory_order_relaxed);
        // the early logits of row i (64-bit words) live in the row's (still unused) unweighted-output block: the exact logits own `scores`
        a.early_logits = r->rawdots; a.early_stride = wv.top_k * wv.hidden;
        RowsK front = k;
        front.plan = nullptr;              // (the front launch names its assignments itself: the work items are written inside it)
        const uint32_t groups = wv.ffn / 32U;
        const bool large = 2ULL * wv.ffn * moe_row_bytes(wv.gate_type, wv.hidden) > kFrontLoneBytes;
        const uint32_t helpers = !large ? 0U : groups < kFrontHelpers / rows ? groups : kFrontHelpers / rows;
        const FrontBlocks nb{rows * ((p->experts + kEarlyExperts - 1U) / kEarlyExperts), a.quant_blocks, rows * ((p->experts + kSideExperts - 1U) / kSideExperts), helpers};
        const uint32_t blocks = nb.early + nb.prologue + nb.side + items * groups + rows * helpers;
        if (do_front) {
            const auto launch = [&](auto helped) {
                constexpr bool HELPED = decltype(helped)::value;
                if (a.kind == MI355_INPUT_F32) layer_front_kernel<0, HELPED><<<blocks, 64, 0, st>>>(wv, front, items, a, nb);
                else if (a.kind == MI355_INPUT_F16) layer_front_kernel<1, HELPED><<<blocks, 64, 0, st>>>(wv, front, items, a, nb);
                else layer_front_kernel<2, HELPED><<<blocks, 64, 0, st>>>(wv, front, items, a, nb);
            };
            if (helpers) launch(std::true_type{});
            else launch(std::false_type{});
            STRIX_LAUNCHED("moe layer early routes + gate / up");
        }
        if (do_back) {
            if (launch_down_merge_format(wv, k, rows, items, form, st)) {
            } else if (wv.top_k <= kDownMergeSlots) launch_down_merge(wv, k, rows, items, form, st);
            else launch_down_merge_quad(wv, k, rows, items, form, st);
            STRIX_LAUNCHED("moe layer experts + combine");
        }
        return MI355_OK;
    }
    if (do_front) {
        launch_route_logits(a, st);
        STRIX_LAUNCHED("moe layer router");
    }
    // the fused router planned one item per routed assignment (and one per four rows of an always-on expert)
    if (p->shared_experts) {       // items of up to four rows: the narrow matrix-core sweeps
        if (do_front) {
            launch_project(wv, layer_rows(), rows, items, st, true);
            STRIX_LAUNCHED("moe layer gate / up");
        }
        if (!do_back) return MI355_OK;
        launch_down(wv, layer_rows(), rows, items, st, true);
        STRIX_LAUNCHED("moe layer experts");
        return enqueue_merge(w, r, rows, form, stream, p->shared_experts);
    }
    if (do_front) launch_project(wv, layer_rows(), rows, items, st);
    if (!do_back) return MI355_OK;
    // down rows and the combine in one launch (the fused router's plan: one item per assignment, in assignment order).
    // A workgroup of that kernel fills a compute unit's LDS; up to four rounds of them it still beats the staged pair of launches
    // (hidden 3072 / ffn 768, 64 experts top-8: 8 rows 76.3 against 82.4 us, 16 rows 115.8 against 121.6 us)
    if (!quad_sweep(wv, rows) && wv.down_type == MI355_TYPE_Q4_K && wv.experts > 1U && wv.top_k <= kDownMergeSlots && wv.hidden % 64U == 0 &&
        (wv.hidden / 64U) * rows <= 4U * compute_units()) {
        launch_down_merge(wv, layer_rows(), rows, items, form, st);
        STRIX_LAUNCHED("moe layer experts + combine");
        return MI355_OK;
    }
    if (quad_sweep(wv, rows) && wv.down_type == MI355_TYPE_Q4_K && wv.top_k <= kDownMergeSlots && wv.hidden % kQuadRows == 0 && rows <= 65535U) {
        launch_down_merge_quad(wv, layer_rows(), rows, items, form, st);
        STRIX_LAUNCHED("moe layer experts + combine");
        return MI355_OK;
    }
    if (launch_down_merge_format(wv, layer_rows(), rows, items, form, st)) {
        STRIX_LAUNCHED("moe layer experts + combine");
        return MI355_OK;
    }
    launch_down(wv, layer_rows(), rows, items, st);
    STRIX_LAUNCHED("moe layer experts");
    return enqueue_merge(w, r, rows, form, stream, p->shared_experts);
}
}  // namespace

extern "C" {

void mi355_debug_early_route_perturb(uint32_t amount) { g_early_perturb.store(amount, std::memory_order_relaxed); }
void mi355_debug_down_merge_flat(uint32_t on) { g_down_merge_flat.store(on != 0, std::memory_order_relaxed); }

int32_t mi355_moe_enqueue_layer(const mi355_route_policy* p, const float* router_weight, const float* logit_bias, float* scores,
                                const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream) {
    return enqueue_layer(p, router_weight, logit_bias, scores, LayerNorm{false, nullptr, 0.0F, nullptr}, w, r, rows, form, stream);
}

int32_t mi355_moe_enqueue_layer_front(const mi355_route_policy* p, const float* router_weight, const float* logit_bias, float* scores,
                                      const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream) {
    return enqueue_layer(p, router_weight, logit_bias, scores, LayerNorm{false, nullptr, 0.0F, nullptr}, w, r, rows, form, stream, kLayerFront);
}

int32_t mi355_moe_enqueue_layer_back(const mi355_route_policy* p, const float* router_weight, const float* logit_bias, float* scores,
                                     const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream) {
    return enqueue_layer(p, router_weight, logit_bias, scores, LayerNorm{false, nullptr, 0.0F, nullptr}, w, r, rows, form, stream, kLayerBack);
}

int32_t mi355_moe_enqueue_layer_normed(const mi355_route_policy* p, const float* router_weight, const float* logit_bias, float* scores,
                                       const float* norm_weight, float norm_eps, float* normed, const mi355_moe_weights* w, const mi355_moe_rows* r,
                                       uint32_t rows, uint32_t form, mi355_stream stream) {
    return enqueue_layer(p, router_weight, logit_bias, scores, LayerNorm{true, norm_weight, norm_eps, normed}, w, r, rows, form, stream);
}

}  // extern "C"
namespace {
// What the prefill kernels see of the caller's rows: dense bundles and the strided PrefillRows views fill it alike.
struct PrefillViews {
    const void* input; uint64_t input_stride;
    RoutesView routes;
    uint32_t* status; uint64_t status_rs;
    uint32_t* job_status;
    float* rawdots; uint64_t rawdots_rs;          // rawdots_rs == 0: dense [assignment][hidden]
    uint32_t rawdots_bf16;
    uint32_t* plan;
    void* h_f16;
};
// expert plan, sub-block sums of the input rows, gate / up + SwiGLU, down rows. check: the routes' check and the status words ride with the
// sums (null: they are already written)
int32_t enqueue_prefill_core(const mi355_moe_weights& wv, const PrefillViews& v, uint32_t rows, hipStream_t st, const RouteCheck* check = nullptr) {
    const uint32_t assignments = rows * wv.top_k, split = prefill_split(wv, assignments), bound = plan_item_bound(wv.experts, assignments, split);
    const PlanArgs plan{v.routes, wv.experts, assignments, split, bound, v.plan};
    PrefillArgs a{};
    a.top_k = wv.top_k; a.exp_kind = wv.exp_kind; a.swiglu_limit = wv.swiglu_limit; a.x = static_cast<const uint8_t*>(v.input); a.x_stride = v.input_stride;
    uint8_t* ws = static_cast<uint8_t*>(v.h_f16);
    a.h = reinterpret_cast<_Float16*>(ws); a.h_lo = reinterpret_cast<_Float16*>(ws + pf_h_plane_bytes(assignments, wv.ffn));
    a.h_sums = ws + pf_h_bytes(assignments, wv.ffn);
    uint8_t* x_sums = a.h_sums + static_cast<size_t>(assignments) * pf_sum_row_bytes(wv.ffn);
    a.x_sums = x_sums;
    a.rawdots = v.rawdots; a.rawdots_rs = v.rawdots_rs; a.rawdots_bf16 = v.rawdots_bf16; a.plan = v.plan; a.experts = wv.experts; a.assignments = assignments;
    a.status = v.status; a.status_rs = v.status_rs; a.job_status = v.job_status; a.items = bound;
    launch_prefill_products(wv, a, rows, x_sums, check, plan, plan_items_at(wv.experts, assignments), plan_order_at(wv.experts), st);
    STRIX_LAUNCHED("moe prefill f16");
    return MI355_OK;
}
}  // namespace
extern "C" {

int32_t mi355_moe_enqueue_prefill_f16(const mi355_moe_weights* w, const mi355_moe_rows* r, uint32_t rows, uint32_t form, mi355_stream stream) {
    mi355_moe_weights wv;
    if (const int32_t rc = check_moe(w, r, rows, wv, kPrefillClass)) return rc;
    STRIX_REQUIRE(form <= MI355_COMBINE_NONE, "moe prefill: unknown combine form");
    STRIX_REQUIRE(r->input && r->input_kind == MI355_INPUT_F16, "moe prefill: the fp16 form takes fp16 input rows");
    STRIX_REQUIRE(r->input_stride % 16U == 0 && aligned(r->input, 16), "moe prefill: input rows must be 16-byte aligned");
    STRIX_REQUIRE(r->h_f16 && aligned(r->h_f16, 16), "moe prefill: h_f16 workspace is null or misaligned");
    STRIX_REQUIRE(rows <= 65535U, "moe prefill: at most 65535 rows per call");
    STRIX_REQUIRE(wv.hidden % 128U == 0 && wv.ffn % 64U == 0, "moe prefill: hidden must be a multiple of 128, ffn of 64");
    hipStream_t st = hs(stream);
    const PrefillViews v{r->input, r->input_stride, dense_routes(r->routes, wv.top_k), r->status, 4, r->job_status, r->rawdots, 0, 0U, r->plan, r->h_f16};
    const RouteCheck check = route_check(wv, *r);
    if (const int32_t rc = enqueue_prefill_core(wv, v, rows, st, &check)) return rc;
    if (form == MI355_COMBINE_NONE) return MI355_OK;
    return mi355_moe_enqueue_merge(w, r, rows, form, stream);
}

int32_t mi355_swiglu_quantize(const float* gate, const float* up, uint32_t rows, uint32_t ffn, uint32_t exp_kind, float swiglu_limit,
                              int8_t* codes, float* deltas, int32_t* sums, float* h_out, uint32_t* status, mi355_stream stream) {
    STRIX_REQUIRE(ffn % 32U == 0, "swiglu: ffn must be a multiple of 32");
    STRIX_REQUIRE(exp_kind <= MI355_EXP_DECLARED, "swiglu: unknown exp kind");
    if (swiglu_limit == 0.0F) swiglu_limit = INFINITY;
    STRIX_REQUIRE(swiglu_limit > 0.0F, "swiglu: swiglu_limit must be +infinity (none) or finite and positive");
    if (rows == 0 || ffn == 0) return MI355_OK;
    STRIX_REQUIRE(gate && up && codes && deltas && sums, "swiglu: null pointer");
    STRIX_REQUIRE(rows <= 65535U, "swiglu: at most 65535 rows per call");
    swiglu_quantize_kernel<<<dim3((ffn / 32U + 7U) / 8U, rows), 256, 0, hs(stream)>>>(gate, up, ffn, exp_kind, swiglu_limit, codes, deltas, sums, h_out, status, nullptr);
    STRIX_LAUNCHED("swiglu_quantize");
    return MI355_OK;
}

// ------------------------------------------------------------------------------------------------------------------
// mi355_moe_enqueue_layer for callers that cannot allocate: every work buffer of the layer (router scores, the A8 images
// of the input and of h, the expert plan, the unweighted down outputs, the job status word) lives in a file-scope device
// array of a fixed size instead of caller memory. Each device holds its own copy of that array; its address on a device is
// looked up once (hipGetSymbolAddress with that device current) and kept, and only that address - never the array's name -
// is handed to kernels.
namespace {
constexpr uint32_t kStaticRows = 16, kStaticTopK = 8, kStaticHidden = 8192, kStaticFfn = 4096, kStaticExperts = 1024;
constexpr uint32_t kStaticAssignments = kStaticRows * kStaticTopK;
constexpr size_t align256(size_t v) { return (v + 255U) & ~static_cast<size_t>(255U); }
constexpr size_t kStaticPlanAt = 0;
constexpr size_t kStaticJobAt = kStaticPlanAt + align256(4U * static_cast<size_t>(plan_words_total(kStaticExperts, kStaticAssignments)));
constexpr size_t kStaticScoresAt = kStaticJobAt + 256U;
constexpr size_t kStaticCodesAt = kStaticScoresAt + align256(4U * static_cast<size_t>(kStaticRows) * kStaticExperts);
constexpr size_t kStaticDeltasAt = kStaticCodesAt + align256(static_cast<size_t>(kStaticRows) * kStaticHidden);
constexpr size_t kStaticSumsAt = kStaticDeltasAt + align256(4U * static_cast<size_t>(kStaticRows) * (kStaticHidden / 32U));
constexpr size_t kStaticDownCodesAt = kStaticSumsAt + align256(4U * static_cast<size_t>(kStaticRows) * (kStaticHidden / 32U));
constexpr size_t kStaticDownDeltasAt = kStaticDownCodesAt + align256(static_cast<size_t>(kStaticAssignments) * kStaticFfn);
constexpr size_t kStaticDownSumsAt = kStaticDownDeltasAt + align256(4U * static_cast<size_t>(kStaticAssignments) * (kStaticFfn / 32U));
constexpr size_t kStaticRawdotsAt = kStaticDownSumsAt + align256(4U * static_cast<size_t>(kStaticAssignments) * (kStaticFfn / 32U));
constexpr size_t kStaticBytes = kStaticRawdotsAt + align256(4U * static_cast<size_t>(kStaticAssignments) * kStaticHidden);    // about 5.1 MB
}  // namespace
static __device__ __align__(256) unsigned char scratch[kStaticBytes];     // zero at load: the plan's ticket words start at zero
namespace {
std::atomic<unsigned char*> g_scratch_of_device[64];
// the array's address on the current device (looked up on the first call there); nullptr with the reason in g_error
unsigned char* scratch_on_current_device() {
    int device = -1;
    const hipError_t e0 = hipGetDevice(&device);
    if (e0 != hipSuccess) { hip_fail(e0, "static workspace: hipGetDevice"); return nullptr; }
    if (device < 0 || device >= 64) { fail(MI355_E_UNSUPPORTED, "static workspace: device ordinal beyond 63"); return nullptr; }
    unsigned char* known = g_scratch_of_device[device].load(std::memory_order_acquire);
    if (known) return known;
    void* found = nullptr;
    const hipError_t e1 = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch));
    if (e1 != hipSuccess || !found) { hip_fail(e1, "static workspace: hipGetSymbolAddress"); return nullptr; }
    g_scratch_of_device[device].store(static_cast<unsigned char*>(found), std::memory_order_release);   // (a racing first call stores the same address)
    return static_cast<unsigned char*>(found);
}
__global__ __launch_bounds__(256) void zero_words_kernel(uint32_t* words, uint32_t count) {
    const uint32_t i = blockIdx.x * 256U + threadIdx.x;
    if (i < count) words[i] = 0U;
}
// The plan words every launch expects to find zero and leaves zero (tickets, arrival counts, tags, the epoch): all zero is the
// state of a freshly loaded library. A kernel store, so that the call may sit inside a captured graph.
int32_t static_plan_reset(unsigned char* ws, hipStream_t st) {
    zero_words_kernel<<<(kPlanOffsetsAt - kPlanTicketsAt + 255U) / 256U, 256, 0, st>>>(reinterpret_cast<uint32_t*>(ws + kStaticPlanAt) + kPlanTicketsAt,
                                                                                  kPlanOffsetsAt - kPlanTicketsAt);
    STRIX_LAUNCHED("static workspace reset");
    return MI355_OK;
}
}  // namespace

int32_t mi355_static_workspace_prepare(mi355_stream stream) {
    unsigned char* ws = scratch_on_current_device();
    if (!ws) return g_error.rfind("static workspace: device", 0) == 0 ? MI355_E_UNSUPPORTED : MI355_E_HIP;
    return static_plan_reset(ws, hs(stream));
}

int32_t mi355_moe_enqueue_layer_static(const mi355_route_policy* p, const float* router_weight, const float* logit_bias,
                                       const mi355_moe_weights* w, const void* input, uint32_t input_kind, uint64_t input_stride,
                                       uint32_t rows, uint32_t* routes, float* route_weights, uint32_t* status, const float* base,
                                       float* output, uint64_t output_stride, uint32_t form, mi355_stream stream) {
    STRIX_REQUIRE(p && w, "moe layer (static workspace): null policy or weights");
    STRIX_REQUIRE(rows >= 1U && rows <= kStaticRows, "moe layer (static workspace): rows must be within 1..16");
    STRIX_REQUIRE(w->top_k >= 1U && w->top_k <= kStaticTopK, "moe layer (static workspace): top_k must be within 1..8");
    STRIX_REQUIRE(w->hidden <= kStaticHidden && w->ffn <= kStaticFfn && w->experts <= kStaticExperts,
                  "moe layer (static workspace): hidden <= 8192, ffn <= 4096 and experts <= 1024 are the limits of the built-in workspace");
    STRIX_REQUIRE(routes && route_weights && status && output && input, "moe layer (static workspace): null row view");
    unsigned char* ws = scratch_on_current_device();
    if (!ws) return g_error.rfind("static workspace: device", 0) == 0 ? MI355_E_UNSUPPORTED : MI355_E_HIP;
    mi355_moe_rows r{};
    r.input = input; r.input_kind = input_kind; r.input_stride = input_stride;
    r.routes = routes; r.route_weights = route_weights; r.status = status; r.base = base; r.output = output; r.output_stride = output_stride;
    r.plan = reinterpret_cast<uint32_t*>(ws + kStaticPlanAt);
    r.job_status = reinterpret_cast<uint32_t*>(ws + kStaticJobAt);
    r.codes = reinterpret_cast<int8_t*>(ws + kStaticCodesAt);
    r.deltas = reinterpret_cast<float*>(ws + kStaticDeltasAt);
    r.sums = reinterpret_cast<int32_t*>(ws + kStaticSumsAt);
    r.down_codes = reinterpret_cast<int8_t*>(ws + kStaticDownCodesAt);
    r.down_deltas = reinterpret_cast<float*>(ws + kStaticDownDeltasAt);
    r.down_sums = reinterpret_cast<int32_t*>(ws + kStaticDownSumsAt);
    r.rawdots = reinterpret_cast<float*>(ws + kStaticRawdotsAt);
    const int32_t rc = mi355_moe_enqueue_layer(p, router_weight, logit_bias, reinterpret_cast<float*>(ws + kStaticScoresAt), w, &r, rows, form, stream);
    // a launch that failed part-way (MI355_E_HIP) may have left counters of the shared plan half-way: put them back to zero for the
    // next call (an admission failure enqueued nothing)
    if (rc == MI355_E_HIP) {
        const std::string first = g_error;
        (void)static_plan_reset(ws, hs(stream));
        g_error = first;
    }
    return rc;
}

}  // extern "C"

#include "a8_contract.hpp"
#include "rows_forms.hpp"
#include "combine_forms.hpp"
#include "shared_gate.hpp"
#include "gguf_reader.hpp"
