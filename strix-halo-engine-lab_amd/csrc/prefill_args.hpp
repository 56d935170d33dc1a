// What the launches of the fp16 prefill form share with the entry points that fill it: the argument block and the workspace layout.
#pragma once
#include "mi355_strix.h"

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace strix950 {

constexpr uint32_t kPfTile = 128;                 // weight rows and tokens per workgroup tile; the most rows of a plan item
constexpr uint32_t kPfFewRows = 32;               // the most rows of an item of the four-wave form
// sub-block sums of a row: two fp16 planes (hi, lo) of `pf_sum_slots(k)` halves each (copied 16 at a time; the slots past k / 32 hold nothing and are never multiplied)
__host__ __device__ constexpr uint32_t pf_sum_slots(uint32_t k) { return (k / 32U + 15U) & ~15U; }
__host__ __device__ constexpr size_t pf_sum_row_bytes(uint32_t k) { return 4U * static_cast<size_t>(pf_sum_slots(k)); }
// bytes of the fp16 workspace: h [assignments][ffn], sums of h [assignments], sums of the input rows [rows]
// (two fp16 planes: h = hi + lo)
// (one plane holds a tile of 128 rows more than the assignments: the down kernel reads whole tiles of rows)
__host__ __device__ constexpr size_t pf_h_plane_bytes(uint32_t assignments, uint32_t ffn) { return 2U * (static_cast<size_t>(assignments) + 128U) * ffn; }
__host__ __device__ constexpr size_t pf_h_bytes(uint32_t assignments, uint32_t ffn) { return 2U * pf_h_plane_bytes(assignments, ffn); }
__host__ __device__ constexpr size_t pf_workspace_bytes(uint32_t hidden, uint32_t ffn, uint32_t rows, uint32_t top_k) {
    return pf_h_bytes(rows * top_k, ffn) + static_cast<size_t>(rows) * top_k * pf_sum_row_bytes(ffn) + static_cast<size_t>(rows) * pf_sum_row_bytes(hidden);
}

struct PrefillArgs {
    const uint8_t* wa; const uint8_t* wb;         // MODE 0: gate, up; MODE 1: down (wb unused)
    uint64_t expert_stride, row_stride;           // bytes
    uint32_t k;                                   // K = hidden (MODE 0) or ffn (MODE 1), multiple of 256
    uint32_t features;                            // ffn (MODE 0) or hidden (MODE 1)
    uint32_t top_k, exp_kind;
    float swiglu_limit;                           // the clamp trait of the SwiGLU epilogue (+infinity: none)
    const uint8_t* x; uint64_t x_stride;          // MODE 0: fp16 token rows (bytes); MODE 1: unused
    _Float16* h;                                  // [assignments in plan order][ffn] fp16: written by MODE 0, read by MODE 1
    _Float16* h_lo;                               // the same shape: fp16(h - fp16(h)), so that hi + lo carries h to 22 bits
    uint8_t* h_sums;                              // [assignments in plan order] sub-block sums of h: written by MODE 0, read by MODE 1
    const uint8_t* x_sums;                        // [rows] sub-block sums of the input rows (MODE 0)
    float* rawdots;                               // MODE 1: [assignment][hidden]
    const uint32_t* plan; uint32_t experts, assignments;
    uint32_t* status; uint32_t* job_status;
    uint32_t tiles, items, units;                 // feature tiles per item, item bound of the launch, tiles * items rounded up to 8 items
    uint64_t status_rs, rawdots_rs;               // bytes between the rows of status / rawdots; rawdots_rs == 0: dense [assignment][features]
    uint32_t rawdots_bf16;                        // MODE 1: every unweighted output is stored once rounded to bfloat16 (as an fp32 value)
};

}  // namespace strix950
