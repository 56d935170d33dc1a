// Router logits of batches past the decode sizes on the fp32 matrix cores. v_mfma_f32_16x16x4_f32 computes every output as four fused
// multiply-adds in ascending k, each rounded once to nearest even, subnormals kept - the reference's ascending fma chain, bit for bit
// (checked over random, wide-range, subnormal and signed-zero operands) -, so a chain of hidden / 4 of them is the chain of
// tests/hip_moe_route_launcher_tests.hip:281-330 for 16 rows x 16 experts at once.
//
// One wave per 16 rows x 16 experts. Its operands come global -> LDS in blocks of 32 features through a ring of its own (a wave that loads
// them to registers in operand order touches 16 rows with 16 neighbouring lanes: 64 separate accesses per instruction, 77 cycles each,
// 34 us a launch), 16-byte pieces with eight (four) neighbouring lanes on a row, piece p of row i at position p ^ i's low bits so that
// eight rows read different banks. Lane (i, q) then reads feature 4 t + q of row i and of expert i for step t of
// the chain with one 32-bit LDS read each (16-byte reads and a transpose between the lanes cost 16 half-rate vector operations per
// eight steps, which the fp32 matrix instruction does not overlap with: 22 us a launch). Bound by the chain, 13.4 ns per 4 features.
// Measured at hidden 2048, 128 experts: 40 and 1000 rows 100 -> 15 and 17 us; 4096 rows, hidden 4096, 256 experts: 221 -> 110 us (lane-wise fma
// chains on tiles of 64 rows x 64 experts before, of which a batch of 40 rows gave two workgroups).
#pragma once
#include "route_wave.hpp"

#include <type_traits>

namespace strix950 {

template <int KIND> constexpr uint32_t route_block_copies() { return KIND == 0 ? 4U : 3U; }      // 2 of the experts, 2 (fp32) or 1 of the rows
template <int KIND, int DEPTH> constexpr uint32_t route_ring_bytes() { return 1024U * route_block_copies<KIND>() * DEPTH; }

// 16 bytes per lane, global -> LDS (lane l lands at lds_at + 16 l), as a plain instruction: arrival is awaited by count
__device__ __forceinline__ void route_copy16(const void* src, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_at), "v"(src) : "memory", "m0");
}

template <int KIND, int DEPTH, uint32_t WAVES>
__global__ __launch_bounds__(64 * WAVES) void route_mma_kernel(RouteArgs a) {
    constexpr uint32_t COPIES = route_block_copies<KIND>(), SLOT = 1024U * COPIES;
    __shared__ __attribute__((aligned(16))) uint8_t ring[WAVES * route_ring_bytes<KIND, DEPTH>()];
    typedef __attribute__((address_space(3))) uint8_t lds_byte;
    typedef const __attribute__((address_space(3))) uint32_t lds_u32;
    typedef const __attribute__((address_space(3))) uint16_t lds_u16;
    typedef const __attribute__((address_space(3))) float lds_f32;
    const uint32_t lane = threadIdx.x & 63U, i = lane & 15U, q = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r0 = blockIdx.y * 16U, e0 = (blockIdx.x * WAVES + wave) * 16U;
    if (e0 >= a.p.experts) return;
    const uint32_t base = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte*)ring)) + wave * route_ring_bytes<KIND, DEPTH>());
    // copier role: lane l of a copy of eight 128-byte rows (fp16 / bf16 activations: sixteen 64-byte rows)
    const auto row_of = [&](uint32_t r) { return a.x + (r0 + r < a.rows ? r0 + r : a.rows - 1U) * a.x_stride; };
    const auto expert_of = [&](uint32_t e) { return a.wr + static_cast<size_t>(e0 + e < a.p.experts ? e0 + e : a.p.experts - 1U) * a.hidden; };
    const uint8_t* src[COPIES];
    const uint32_t piece8 = (lane & 7U) ^ (lane >> 3);
    src[0] = reinterpret_cast<const uint8_t*>(expert_of(lane >> 3)) + 16U * piece8;
    src[1] = reinterpret_cast<const uint8_t*>(expert_of(8U + (lane >> 3))) + 16U * piece8;
    if constexpr (KIND == 0) {
        src[2] = row_of(lane >> 3) + 16U * piece8;
        src[3] = row_of(8U + (lane >> 3)) + 16U * piece8;
    } else src[2] = row_of(lane >> 2) + 16U * ((lane & 3U) ^ ((lane >> 3) & 3U));
    const uint32_t blocks = a.hidden / 32U;
    const auto issue = [&](uint32_t at) {               // (past the end: the last block again, never read; the counts stay the same)
        const uint32_t k = 32U * (at < blocks ? at : blocks - 1U), slot = __builtin_amdgcn_readfirstlane(base + (at % DEPTH) * SLOT);
#pragma unroll
        for (uint32_t c = 0; c < COPIES; ++c) route_copy16(src[c] + (c < 2U || KIND == 0 ? 4U : 2U) * k, slot + 1024U * c);
    };
    // step t of half h: LDS bytes of the lane's expert and row value inside a slot
    uint32_t w_at[8], x_at[8];
#pragma unroll
    for (uint32_t t = 0; t < 8U; ++t) {
        w_at[t] = base + 128U * i + 16U * (t ^ (i & 7U)) + 4U * q;
        if constexpr (KIND == 0) x_at[t] = w_at[t] + 2048U;
        else x_at[t] = base + 2048U + 64U * i + 16U * ((t >> 1) ^ ((i >> 1) & 3U)) + 2U * ((4U * t + q) & 7U);
    }
    struct Block { float w[8]; uint32_t x[8]; };
    const auto read = [&](Block& b, uint32_t slot) {
#pragma unroll
        for (uint32_t t = 0; t < 8U; ++t) {
            b.w[t] = *(lds_f32*)(uintptr_t)(w_at[t] + slot * SLOT);
            if constexpr (KIND == 0) b.x[t] = *(lds_u32*)(uintptr_t)(x_at[t] + slot * SLOT);
            else b.x[t] = *(lds_u16*)(uintptr_t)(x_at[t] + slot * SLOT);
        }
    };
    f32x4 acc = {0.0F, 0.0F, 0.0F, 0.0F};
    const auto chain = [&](const Block& b) {
#pragma unroll
        for (uint32_t t = 0; t < 8U; ++t) {
            const float x = KIND == 0 ? f_of(b.x[t]) : KIND == 1 ? half_bits_to_float(b.x[t]) : f_of(b.x[t] << 16);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x, b.w[t], acc, 0, 0, 0);
        }
    };
#pragma unroll
    for (uint32_t s = 0; s < DEPTH; ++s) issue(s);
    Block now, next;
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES * (DEPTH - 1U)) : "memory");
    read(now, 0);
    const auto step = [&](uint32_t at, uint32_t s, Block& here, Block& ahead) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");          // this block is in registers: its slot is free
        issue(at + DEPTH);
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES * (DEPTH - 1U)) : "memory");
        read(ahead, (s + 1U) % DEPTH);
        chain(here);
    };
    for (uint32_t at = 0; at < blocks; at += DEPTH) {               // (slot s of a turn holds block at + s: the offsets are constants)
#pragma unroll
        for (uint32_t s = 0; s < DEPTH; s += 2U) {
            if (at + s < blocks) step(at + s, s, now, next);
            if (at + s + 1U < blocks) step(at + s + 1U, s + 1U, next, now);
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");     // no copy may land after the wave has given its LDS back
    // lane (i, q): expert i, rows 4 q .. 4 q + 3
    const uint32_t e = e0 + i;
    if (e >= a.p.experts) return;
    const float bias = a.bias ? a.bias[e] : 0.0F;
#pragma unroll
    for (uint32_t t = 0; t < 4U; ++t) {
        const uint32_t r = r0 + 4U * q + t;
        if (r < a.rows) a.scores[static_cast<size_t>(r) * a.p.experts + e] = a.bias ? acc[t] + bias : acc[t];
    }
}

// While a wave's workgroup finds room beside two others (fp32 rows: beside one), a ring of sixteen blocks (48 KB, 64 KB): a block is chained in
// 107 ns, so eight are 0.9 us ahead, less than a cold fetch takes (hidden 2048, 128 experts, 40 | 333 rows 16.7 | 15.9 -> 14.7 | 14.4 us; hidden 6144,
// 160 experts, 17 rows 39.3 -> 36.5; 1008 waves of hidden 2048 17.3 | 30.0). Else four waves a workgroup: a ring of eight where one workgroup per
// compute unit holds the launch, of four (two or three workgroups share a unit) beyond.
inline void launch_route_mma(const RouteArgs& a, uint32_t compute_units, hipStream_t st) {
    const uint32_t rows = (a.rows + 15U) / 16U, experts = (a.p.experts + 15U) / 16U;
    const uint64_t waves = static_cast<uint64_t>(rows) * experts, units = compute_units;
    const auto launch = [&](auto depth, auto per) {
        constexpr int DEPTH = decltype(depth)::value;
        constexpr uint32_t WAVES = decltype(per)::value;
        const dim3 grid((experts + WAVES - 1U) / WAVES, rows);
        if (a.kind == MI355_INPUT_F32) route_mma_kernel<0, DEPTH, WAVES><<<grid, 64U * WAVES, 0, st>>>(a);
        else if (a.kind == MI355_INPUT_F16) route_mma_kernel<1, DEPTH, WAVES><<<grid, 64U * WAVES, 0, st>>>(a);
        else route_mma_kernel<2, DEPTH, WAVES><<<grid, 64U * WAVES, 0, st>>>(a);
    };
    if (waves <= (a.kind == MI355_INPUT_F32 ? 2U : 3U) * units) launch(std::integral_constant<int, 16>{}, std::integral_constant<uint32_t, 1U>{});
    else if (static_cast<uint64_t>((experts + 3U) / 4U) * rows <= units) launch(std::integral_constant<int, 8>{}, std::integral_constant<uint32_t, 4U>{});
    else launch(std::integral_constant<int, 4>{}, std::integral_constant<uint32_t, 4U>{});
}

}  // namespace strix950
