// A8 image of activation rows: one workgroup per row, a thread quantises eight neighbouring values, four threads a group of 32.
// Reference: src/cpu/core/reference.cpp:35-55.
// Bound by latency (one row) or by the rows' bytes (many): 128-bit loads, 64-bit code stores, and the row's status word leaves in one
// store of the workgroup, so a caller that has no earlier bits in it needs no clearing launch in front.
#pragma once
#include "device_math.hpp"
#include "mi355_strix.h"

namespace strix950 {

// How the row's status word is written: not at all, bits ORed in, or stored (the whole word).
enum A8Status : uint32_t { kA8StatusNone = 0, kA8StatusOr = 1, kA8StatusStore = 2 };

struct A8RowArgs {
    const uint8_t* x; uint64_t x_stride; uint32_t width;
    int8_t* codes; float* deltas; int32_t* sums; uint32_t* status;
    uint32_t status_mode, vec;           // vec: rows are 16-byte aligned, codes 8-byte: 128-bit loads, 64-bit stores
    // the dense A8 profile's rule for a group that holds a non-finite value (src/hip_q8_rows_gemv.hpp:1157-1161,1232-1250): its delta
    // is the canonical NaN 0x7fc00000 and its codes are 0, so that every product over the group is NaN
    uint32_t nan_delta;
};

template <int KIND>
__device__ __forceinline__ void load_activation8(const uint8_t* row, uint32_t i, bool vec, float (&v)[8]) {
    if (vec) {
        if constexpr (KIND == 0) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(row + 4U * i), b = *reinterpret_cast<const f32x4*>(row + 4U * i + 16U);
#pragma unroll
            for (int q = 0; q < 4; ++q) { v[q] = a[q]; v[4 + q] = b[q]; }
        } else {
            const u32x4 a = *reinterpret_cast<const u32x4*>(row + 2U * i);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (KIND == 1) { v[2 * q] = half_bits_to_float(a[q] & 0xffffU); v[2 * q + 1] = half_bits_to_float(a[q] >> 16); }
                else { v[2 * q] = f_of(a[q] << 16); v[2 * q + 1] = f_of(a[q] & 0xffff0000U); }
            }
        }
    } else {
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) v[q] = load_activation<KIND>(row, i + q);
    }
}

// The row's image by the first `threads` (a multiple of 64) of the calling workgroup; returns non-zero in the threads of a group with a
// non-finite value.
template <int KIND>
__device__ __forceinline__ int a8_row(const A8RowArgs& a, uint32_t r, uint32_t threads) {
    const uint8_t* row = a.x + r * a.x_stride;
    int8_t* codes = a.codes + static_cast<size_t>(r) * a.width;
    const uint32_t groups = a.width / 32U;
    int any_bad = 0;
    for (uint32_t i = threadIdx.x * 8U; i < a.width; i += threads * 8U) {          // (a group's four threads leave the loop together)
        float v[8];
        load_activation8<KIND>(row, i, a.vec != 0, v);
        float amax = __builtin_fabsf(v[0]);
        int bad = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            amax = __builtin_fmaxf(amax, __builtin_fabsf(v[q]));
            bad |= finite_f(v[q]) ? 0 : 1;
        }
        amax = __builtin_fmaxf(amax, xor1_f(amax)); amax = __builtin_fmaxf(amax, xor2_f(amax));
        bad |= xor1_i(bad); bad |= xor2_i(bad);
        const bool tiny = amax > 0.0F && amax < 0x1p-119F, poison = bad && a.nan_delta;
        const float delta = (amax == 0.0F || tiny) ? 1.0F : amax / 127.0F;
        uint32_t packed[2] = {0, 0};
        int sum = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int code = poison ? 0 : a8_code(v[q], delta, tiny);
            sum += code;
            packed[q >> 2] |= (static_cast<uint32_t>(code) & 0xffU) << (8 * (q & 3));
        }
        if (a.vec) *reinterpret_cast<uint2*>(codes + i) = make_uint2(packed[0], packed[1]);
        else
#pragma unroll
            for (int q = 0; q < 8; ++q) codes[i + q] = static_cast<int8_t>(packed[q >> 2] >> (8 * (q & 3)));
        sum += xor1_i(sum); sum += xor2_i(sum);
        if ((threadIdx.x & 3U) == 0U) {
            const size_t at = static_cast<size_t>(r) * groups + i / 32U;
            a.deltas[at] = poison ? f_of(0x7fc00000U) : delta;
            if (a.sums) a.sums[at] = sum;
        }
        any_bad |= bad;
    }
    return any_bad;
}

template <int KIND>
__global__ __launch_bounds__(1024) void a8_rows_kernel(A8RowArgs a) {
    const uint32_t r = blockIdx.x;
    const int bad = a8_row<KIND>(a, r, blockDim.x);
    if (a.status_mode == kA8StatusNone) return;
    const uint32_t bits = __syncthreads_or(bad) ? static_cast<uint32_t>(MI355_STATUS_NONFINITE_ACTIVATION) : 0U;
    if (threadIdx.x == 0) {
        if (a.status_mode == kA8StatusStore) a.status[r] = bits;
        else if (bits) atomicOr(&a.status[r], bits);
    }
}

// one pass of the row where it fits a workgroup of 1024 threads
inline uint32_t a8_row_threads(uint32_t width) {
    const uint32_t waves = (width / 8U + 63U) / 64U;
    return 64U * (waves < 16U ? waves : 16U);
}

}  // namespace strix950
