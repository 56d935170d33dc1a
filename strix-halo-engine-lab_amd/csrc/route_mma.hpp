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
// Measured with the selection behind it, LDS reads in front of a block's products and address arithmetic between them -> reads between the
// products, vector operations in front: hidden 2048, 128 experts, 40 | 333 | 1000 rows 19.0 | 19.3 | 20.3 -> 17.1 | 17.4 | 18.3 us; 17 rows of hidden 6144, 160 experts
// 42.3 -> 36.9; 100 of 4096, 64 experts 29.8 -> 26.0; 4096 rows of 4096, 256 experts 110 -> 98. (Lane-wise fma chains on tiles of 64 rows x 64
// experts, of which a batch of 40 rows gives two workgroups, take 100 us for the first.)
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

// the same from a base of the wave and a byte offset per lane
__device__ __forceinline__ void route_copy16_at(uint64_t base, uint32_t offset, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_at), "v"(offset), "s"(base) : "memory", "m0");
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
    const uint32_t piece8 = (lane & 7U) ^ (lane >> 3), last = a.p.experts - 1U - e0;
    // experts: the wave's first one, and bytes from there (sixteen rows of at most 64 KB)
    const uint64_t w_base = reinterpret_cast<uint64_t>(a.wr + static_cast<size_t>(e0) * a.hidden);
    const uint32_t w_off[2] = {((lane >> 3) < last ? lane >> 3 : last) * 4U * a.hidden + 16U * piece8, (8U + (lane >> 3) < last ? 8U + (lane >> 3) : last) * 4U * a.hidden + 16U * piece8};
    const uint8_t* x_src[COPIES - 2U];
    if constexpr (KIND == 0) {
        x_src[0] = row_of(lane >> 3) + 16U * piece8;
        x_src[1] = row_of(8U + (lane >> 3)) + 16U * piece8;
    } else x_src[0] = row_of(lane >> 2) + 16U * ((lane & 3U) ^ ((lane >> 3) & 3U));
    const uint32_t blocks = a.hidden / 32U;
    // copies of block `at` (past the end: the last block again, never read; the counts stay the same)
    const auto issue_weights = [&](uint32_t at) __attribute__((always_inline)) {
        const uint32_t k = at < blocks ? at : blocks - 1U, slot = __builtin_amdgcn_readfirstlane(base + (at % DEPTH) * SLOT);
#pragma unroll
        for (uint32_t c = 0; c < 2U; ++c) route_copy16_at(w_base + 128ULL * k, w_off[c], slot + 1024U * c);
    };
    const uint8_t* x_next[COPIES - 2U];
    const auto place_rows = [&](uint32_t at) __attribute__((always_inline)) {
        const uint32_t k = at < blocks ? at : blocks - 1U;
#pragma unroll
        for (uint32_t c = 0; c < COPIES - 2U; ++c) x_next[c] = x_src[c] + (KIND == 0 ? 128U : 64U) * k;
    };
    const auto issue_rows = [&](uint32_t at) __attribute__((always_inline)) {
        const uint32_t slot = __builtin_amdgcn_readfirstlane(base + (at % DEPTH) * SLOT);
#pragma unroll
        for (uint32_t c = 0; c < COPIES - 2U; ++c) route_copy16(x_next[c], slot + 2048U + 1024U * c);
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
    const auto read = [&](Block& b, uint32_t slot, uint32_t from, uint32_t to) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t t = from; t < to; ++t) {
            b.w[t] = *(lds_f32*)(uintptr_t)(w_at[t] + slot * SLOT);
            if constexpr (KIND == 0) b.x[t] = *(lds_u32*)(uintptr_t)(x_at[t] + slot * SLOT);
            else b.x[t] = *(lds_u16*)(uintptr_t)(x_at[t] + slot * SLOT);
        }
    };
    f32x4 acc = {0.0F, 0.0F, 0.0F, 0.0F};
#pragma unroll
    for (uint32_t s = 0; s < DEPTH; ++s) { issue_weights(s); place_rows(s); issue_rows(s); }
    Block now, next;
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES * (DEPTH - 1U)) : "memory");
    read(now, 0, 0U, 8U);
    // The vector ALU stands still while an fp32 product runs, and each change from one to the other costs 17 cycles (chain alone 32 cycles a product;
    // with one vector operation in every gap 49, with four 72; with eight conversions in front of eight products 38): a block's vector
    // operations come first, in one run. LDS reads, copies and scalar operations go on beside a product (two reads in every gap 34,
    // sixteen in front of eight products 53), so they stand in the gaps.
    const auto step = [&](uint32_t at, uint32_t s, const Block& here, Block& ahead) __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");          // this block is in registers: its slot is free
        float x[8];
#pragma unroll
        for (uint32_t t = 0; t < 8U; ++t) {
            x[t] = KIND == 0 ? f_of(here.x[t]) : KIND == 1 ? half_bits_to_float(here.x[t]) : f_of(here.x[t] << 16);
            asm volatile("" : "+v"(x[t]));
        }
        place_rows(at + DEPTH);
#pragma unroll
        for (uint32_t c = 0; c < COPIES - 2U; ++c) asm volatile("" : "+v"(x_next[c]));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t t = 0; t < 8U; ++t) {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], here.w[t], acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (t == 0U) issue_weights(at + DEPTH);
            else if (t == 1U) {
                issue_rows(at + DEPTH);
                asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES * (DEPTH - 1U)) : "memory");
            } else if (t < 6U) read(ahead, (s + 1U) % DEPTH, 2U * t - 4U, 2U * t - 2U);
            __builtin_amdgcn_sched_barrier(0);
        }
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

// The same with a second wave that brings the operands: it starts the copies, awaits them, widens fp16 / bf16 rows to fp32 in LDS, four blocks ahead, and meets the
// chaining wave once for those. That one has no vector operation between its products: 35.4 cycles each, where it does everything
// itself 46 (meeting once a block the second wave is the slower one of the two with rows to widen: 43). Logits and selection, one wave -> two: 40 fp16 | fp32 rows of
// hidden 2048, 128 experts 17.0 | 17.9 -> 14.5 | 14.3 us, 333 rows 17.3 -> 14.8; 17 rows of 6144, 160 experts 36.8 -> 29.2; 100 of 4096, 64 experts 26.1 -> 21.0.
template <int KIND, int DEPTH>
__global__ __launch_bounds__(128) void route_mma_pair_kernel(RouteArgs a) {
    constexpr uint32_t COPIES = route_block_copies<KIND>(), SLOT = 1024U * COPIES, TURN = 4U, WIDENED = 2U * TURN;       // blocks from meeting to meeting, blocks of widened rows
    static_assert(DEPTH % WIDENED == 0, "a block's places follow from its place in the ring");
    __shared__ __attribute__((aligned(16))) uint8_t ring[route_ring_bytes<KIND, DEPTH>() + (KIND == 0 ? 0U : 2048U * WIDENED)];
    typedef __attribute__((address_space(3))) uint8_t lds_byte;
    typedef const __attribute__((address_space(3))) float lds_f32;
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
    const uint32_t lane = threadIdx.x & 63U, i = lane & 15U, q = lane >> 4;
    const uint32_t r0 = blockIdx.y * 16U, e0 = blockIdx.x * 16U, blocks = a.hidden / 32U;
    const uint32_t base = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte*)ring)));
    const uint32_t widened = base + route_ring_bytes<KIND, DEPTH>();
    const auto meet = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) != 0U) {
        const auto row_of = [&](uint32_t r) { return a.x + (r0 + r < a.rows ? r0 + r : a.rows - 1U) * a.x_stride; };
        const auto expert_of = [&](uint32_t e) { return reinterpret_cast<const uint8_t*>(a.wr + static_cast<size_t>(e0 + e < a.p.experts ? e0 + e : a.p.experts - 1U) * a.hidden); };
        const uint32_t piece8 = (lane & 7U) ^ (lane >> 3), row = lane >> 2, piece = lane & 3U;
        const uint8_t* src[COPIES];
        src[0] = expert_of(lane >> 3) + 16U * piece8;
        src[1] = expert_of(8U + (lane >> 3)) + 16U * piece8;
        if constexpr (KIND == 0) {
            src[2] = row_of(lane >> 3) + 16U * piece8;
            src[3] = row_of(8U + (lane >> 3)) + 16U * piece8;
        } else src[2] = row_of(row) + 16U * piece;
        const auto issue = [&](uint32_t at) {           // (past the end: the last block again, never read; the counts stay the same)
            const uint32_t k = at < blocks ? at : blocks - 1U, slot = __builtin_amdgcn_readfirstlane(base + (at % DEPTH) * SLOT);
#pragma unroll
            for (uint32_t c = 0; c < COPIES; ++c) route_copy16(src[c] + (c < 2U || KIND == 0 ? 128U : 64U) * k, slot + 1024U * c);
        };
        const auto widen = [&](uint32_t at) {           // blocks at .. at + TURN - 1
            if constexpr (KIND != 0) {
                u32x4 raw[TURN];
#pragma unroll
                for (uint32_t b = 0; b < TURN; ++b) raw[b] = *(lds_u32x4*)(uintptr_t)(base + ((at + b) % DEPTH) * SLOT + 2048U + 16U * lane);
#pragma unroll
                for (uint32_t b = 0; b < TURN; ++b) {
                    f32x4 f[2];
#pragma unroll
                    for (uint32_t n = 0; n < 4U; ++n) {
                        f[n >> 1][2U * (n & 1U)] = KIND == 1 ? half_bits_to_float(raw[b][n] & 0xffffU) : f_of(raw[b][n] << 16);
                        f[n >> 1][2U * (n & 1U) + 1U] = KIND == 1 ? half_bits_to_float(raw[b][n] >> 16) : f_of(raw[b][n] & 0xffff0000U);
                    }
                    const uint32_t to = widened + 2048U * ((at + b) % WIDENED) + 128U * row;
#pragma unroll
                    for (uint32_t n = 0; n < 2U; ++n) *(lds_f32x4*)(uintptr_t)(to + 16U * ((2U * piece + n) ^ (row & 7U))) = f[n];
                }
            }
        };
        for (uint32_t s = 0; s < DEPTH; ++s) issue(s);
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES * (DEPTH - TURN)) : "memory");
        widen(0);
        meet();
        for (uint32_t at = 0; at + TURN <= blocks; at += TURN) {
            asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES * (DEPTH - 2U * TURN)) : "memory");
            widen(at + TURN);
            meet();                                     // blocks at .. at + 3 are in the chaining wave's registers or behind them, the next four in LDS
#pragma unroll
            for (uint32_t b = 0; b < TURN; ++b) issue(at + DEPTH + b);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // no copy may land after the workgroup has given its LDS back
        return;
    }
    // step t: LDS bytes of the lane's expert and row value (feature 4 t + q) inside a slot
    uint32_t w_at[8], x_at[8];
#pragma unroll
    for (uint32_t t = 0; t < 8U; ++t) {
        const uint32_t in = 128U * i + 16U * (t ^ (i & 7U)) + 4U * q;
        w_at[t] = base + in;
        x_at[t] = (KIND == 0 ? base + 2048U : widened) + in;
    }
    struct Block { float w[8], x[8]; };
    const auto read = [&](Block& b, uint32_t s, uint32_t from, uint32_t to) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t t = from; t < to; ++t) {
            b.w[t] = *(lds_f32*)(uintptr_t)(w_at[t] + s * SLOT);
            b.x[t] = *(lds_f32*)(uintptr_t)(x_at[t] + (KIND == 0 ? s * SLOT : (s % WIDENED) * 2048U));
        }
    };
    f32x4 acc = {0.0F, 0.0F, 0.0F, 0.0F};
    Block now, next;
    const auto step = [&](uint32_t s, const Block& here, Block& ahead) __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t t = 0; t < 8U; ++t) {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(here.x[t], here.w[t], acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (t == 0U && s % TURN == TURN - 1U) meet();
            if (t > 0U && t < 5U) read(ahead, (s + 1U) % DEPTH, 2U * t - 2U, 2U * t);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    meet();
    read(now, 0, 0U, 8U);
    for (uint32_t at = 0; at < blocks; at += DEPTH) {               // (slot s of a turn holds block at + s: the offsets are constants)
#pragma unroll
        for (uint32_t s = 0; s < DEPTH; s += 2U) {
            if (at + s < blocks) step(s, now, next);
            if (at + s + 1U < blocks) step(s + 1U, next, now);
        }
    }
    const uint32_t e = e0 + i;
    if (e >= a.p.experts) return;
    const float bias = a.bias ? a.bias[e] : 0.0F;
#pragma unroll
    for (uint32_t t = 0; t < 4U; ++t) {
        const uint32_t r = r0 + 4U * q + t;
        if (r < a.rows) a.scores[static_cast<size_t>(r) * a.p.experts + e] = a.bias ? acc[t] + bias : acc[t];
    }
}

// Two waves a tile while their workgroup finds room beside another (1000 rows of hidden 2048, 128 experts, 504 tiles: one wave 17.7, two 17.4 us; 1500 rows 18.8 | 30).
// Past that, while a wave's workgroup finds room beside two others, a ring of sixteen blocks (48 KB; of fp32 rows 64 KB, which leaves no room for a third): a block is chained in
// 125 ns, so eight are 1 us ahead, less than a cold fetch takes (hidden 2048, 128 experts, 40 | 333 rows 16.7 | 15.9 -> 14.7 | 14.4 us; hidden 6144,
// 160 experts, 17 rows 39.3 -> 36.5; 1008 waves of hidden 2048 17.3 | 30.0, with a block in 140 ns). Else four waves a workgroup: a ring of eight where one workgroup per
// compute unit holds the launch, of four (two or three workgroups share a unit) beyond.
inline void launch_route_mma(const RouteArgs& a, uint32_t compute_units, hipStream_t st) {
    const uint32_t rows = (a.rows + 15U) / 16U, experts = (a.p.experts + 15U) / 16U;
    const uint64_t waves = static_cast<uint64_t>(rows) * experts, units = compute_units;
    const auto launch = [&](auto depth, auto per) {
        constexpr int DEPTH = decltype(depth)::value;
        constexpr uint32_t WAVES = decltype(per)::value;
        const dim3 grid((experts + WAVES - 1U) / WAVES, rows);
        if (a.kind == MI355_INPUT_F32) {
            if constexpr (DEPTH < 16) route_mma_kernel<0, DEPTH, WAVES><<<grid, 64U * WAVES, 0, st>>>(a);
        } else if (a.kind == MI355_INPUT_F16) route_mma_kernel<1, DEPTH, WAVES><<<grid, 64U * WAVES, 0, st>>>(a);
        else route_mma_kernel<2, DEPTH, WAVES><<<grid, 64U * WAVES, 0, st>>>(a);
    };
    if (waves <= 2U * units) {
        const dim3 grid(experts, rows);
        if (a.kind == MI355_INPUT_F32) route_mma_pair_kernel<0, 16><<<grid, 128, 0, st>>>(a);
        else if (a.kind == MI355_INPUT_F16) route_mma_pair_kernel<1, 16><<<grid, 128, 0, st>>>(a);
        else route_mma_pair_kernel<2, 16><<<grid, 128, 0, st>>>(a);
    } else if (a.kind != MI355_INPUT_F32 && waves <= 3U * units) launch(std::integral_constant<int, 16>{}, std::integral_constant<uint32_t, 1U>{});
    else if (static_cast<uint64_t>((experts + 3U) / 4U) * rows <= units) launch(std::integral_constant<int, 8>{}, std::integral_constant<uint32_t, 4U>{});
    else launch(std::integral_constant<int, 4>{}, std::integral_constant<uint32_t, 4U>{});
}

}  // namespace strix950
