// Q4_K x A8 rows (and the reference's other formats of expert rows, below) against 1..32 activation rows at a time: the exact group dots come from the int8 matrix cores, the
// reference's fp32 chain stays on the vector ALU. The sweep below serves dense matrices and the routed
// experts of larger batches (q4k_mma_moe.hpp: gate + up with the SwiGLU / A8 epilogue, and the down rows).
//
// A workgroup (4 wavefronts) owns 32 weight rows. Wavefront p owns the reference's pair accumulator p of those rows
// (sub-blocks 2p and 2p + 1 of every super-block) - the four pair chains of a row are independent, K is never split.
// Per super-block a wavefront issues two v_mfma_i32_32x32x32_i8: operand B = 32 weight rows x the 32 nibbles of one
// sub-block (lane (row j, half h) carries elements 16h .. 16h + 15, expanded to bytes), operand A = 32 activation slots x the
// same 32 codes (lane (slot i, half h) carries codes 16h .. 16h + 15 of its row). Both operands put element k in the same
// register byte, so whatever order the core walks K in, a product pairs weight k with code k; an integer sum has no order.
// The 32 x 32 result leaves lane (j, h) with its row's dots against the slots 8 (v / 4) + 4h + v % 4, v = 0..15; activation
// row a sits in slot v = a / 2 of half h = a % 2, so the lane reads rows h, 2 + h, 4 + h, ... from result registers 0, 1, 2, ...
// and every lane of the wavefront does chain work for NAL = ceil(rows / 2) activation rows.
//
// Chain per (row, activation row, sub-block) - src/cpu/core/routed_expert.cpp:73-108 == src/moe_q4k_a8_contract.cpp:126-140:
//   u = (d * scale) * float(dot); v = (dmin * min) * float(code sum); x = delta * (u - v); acc[p] += x[2p] + x[2p + 1];
//   value = (acc[0] + acc[1]) + (acc[2] + acc[3]).
// delta and code sum depend on (activation row, sub-block) only: every quad of lanes keeps the four values of the wavefront's
// two sub-blocks (delta 2p, delta 2p + 1, sum 2p, sum 2p + 1) in its four lanes and the multiplies take them by quad
// broadcast (a DPP operand, no instruction of its own).
//
// Data path: a stage is one super-block (256 weights) of the 32 rows in 16-byte pieces, an odd number of them from row to row, so that
// sixteen neighbouring rows read sixteen different 16-byte bank groups (the even 14 and 12 of Q6_K and Q5_1: down rows of a layer of 40 rows,
// hidden 2048 / ffn 768 / 128 experts, Q5_1 139 -> 127 us; three calls over a union of 6 x 16 Q6_K rows, 90 -> 78), the 256 codes of every activation row (piece t of row a at
// position (t + a) % 16 of its 16 pieces, which spreads eight rows over the bank groups) and one table piece per row
// (8 deltas, 8 sums). Everything arrives by global_load_lds_dwordx4 into a ring of DEPTH slots shared by the workgroup: a
// wavefront waits for its own copies (counted s_waitcnt vmcnt), the workgroup barrier publishes all of them, and the slot
// consumed before the barrier is refilled after it.
//
// A workgroup runs over consecutive 32-row tiles against the same activation rows, and the ring does not stop between them: the
// copies of the next tile's first stages are in flight while a tile's last stages are multiplied and its values leave. Rows of few
// super-blocks would otherwise pay the start of a ring (the chain from the work item to the first arrival) every few stages.
#pragma once
#include "q4k_pairs.hpp"

#include <type_traits>

namespace strix950 {

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) uint64_t lds_u64;
typedef __attribute__((address_space(3))) uint32_t lds_u32;

constexpr uint32_t kMmaRows = 32;
// Formats of the weight rows: bytes of 256 weights of a row and the 16-byte pieces that hold them (Q6_K: that hold them wherever in a piece
// the 2-byte aligned block starts).
enum MmaFormat { kMmaQ4K, kMmaQ5K, kMmaQ6K, kMmaQ80, kMmaQ51 };
template <int FMT> constexpr uint32_t mma_block_bytes() { return FMT == kMmaQ4K ? 144U : FMT == kMmaQ5K ? 176U : FMT == kMmaQ6K ? 210U : FMT == kMmaQ80 ? 272U : 192U; }
template <int FMT> constexpr uint32_t mma_pieces() { return (mma_block_bytes<FMT>() + 15U) / 16U; }
// pieces from a row to the next one in a ring slot: an odd number, so that the same words of sixteen rows lie in different banks
template <int FMT> constexpr uint32_t mma_pitch() { return mma_pieces<FMT>() | 1U; }
template <int FMT> constexpr uint32_t mma_weight_copies() { return (mma_pitch<FMT>() + 1U) / 2U; }          // 1 KiB = 64 pieces, the last half a wave's
template <int FMT> constexpr uint32_t mma_weight_bytes() { return 16U * mma_pitch<FMT>() * kMmaRows; }
template <int NAL> constexpr uint32_t mma_acts() { return 2U * NAL; }                         // activation slots served (multiple of 4)
template <int NAL> constexpr uint32_t mma_code_copies() { return mma_acts<NAL>() / 4U; }      // 1 KiB = 4 rows x 256 codes
template <int NAL> constexpr uint32_t mma_table_copies() { return (mma_acts<NAL>() + 15U) / 16U; }   // 1 KiB = 16 rows x (8 deltas, 8 sums)
// NM matrices share the activation rows of a sweep (gate and up)
template <int FMT, int NAL, int NM> constexpr uint32_t mma_copies() { return mma_weight_copies<FMT>() * NM + mma_code_copies<NAL>() + mma_table_copies<NAL>(); }
template <int FMT, int NM> constexpr uint32_t mma_codes_at() { return mma_weight_bytes<FMT>() * NM; }
template <int FMT, int NAL, int NM> constexpr uint32_t mma_table_at() { return mma_codes_at<FMT, NM>() + 256U * mma_acts<NAL>(); }
template <int FMT, int NAL, int NM> constexpr uint32_t mma_slot_bytes() { return mma_table_at<FMT, NAL, NM>() + (mma_acts<NAL>() < 16U ? 64U * mma_acts<NAL>() : 1024U * mma_table_copies<NAL>()); }
template <int FMT, int NAL, int NM, int DEPTH, int TEAMS> constexpr uint32_t mma_ring_bytes() { return DEPTH * TEAMS * mma_slot_bytes<FMT, NAL, NM>(); }
template <int NAL, int TEAMS> constexpr uint32_t mma_exchange_floats() { return TEAMS > 1 ? 2U * (TEAMS - 1U) * 4U * NAL * 64U : 1U; }
// The wide form (mma_stage_wide) serves sweeps of 32 activation rows: of Q4_K down rows, and of gate / up rows where it is the faster one (mma_project_wide).
template <int FMT, int NAL> constexpr bool mma_wide() { return NAL == 16 && (FMT == kMmaQ4K || FMT == kMmaQ5K); }
// Wavefronts that sweep a tile together: four (one a pair accumulator), in the wide form four for each matrix.
template <int NM, bool WIDE> constexpr uint32_t mma_waves() { return WIDE ? 4U * NM : 4U; }
template <int NAL, int NM> constexpr uint32_t mma_reduce_floats() { return 4U * NM * NAL * 64U; }

// Workgroup barrier that orders LDS traffic only (__syncthreads() would also wait for every copy in flight, i.e. drain the
// ring at each stage): this wavefront's LDS reads and writes complete, then the barrier; arrivals of copies are awaited by count.
__device__ __forceinline__ void mma_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One global -> LDS copy of 16 bytes per lane (lane l lands at lds_at + 16 l), issued as plain instructions: told about the copy,
// the compiler would hold every later LDS read until all copies in flight have landed. Arrival is awaited by count instead.
__device__ __forceinline__ void mma_copy16(const uint8_t* src, lds_u8* lds_at) {
    const uint32_t at = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds_at)));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(at), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ uint64_t mma_scalar(uint64_t v) {
    return static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32)))) << 32 |
           static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v)));
}
// the same for the lanes of `lanes` only, at least one. Every lane of the wavefront is active around it: the kernels run whole wavefronts,
// and no copy stands behind a condition on the lane. (A copy without a lane may not be counted as an operation in flight.)
__device__ __forceinline__ void mma_copy16_lanes(const uint8_t* src, lds_u8* lds_at, uint64_t lanes) {
    const uint32_t at = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds_at)));
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %2\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b64 exec, -1"
                 : : "s"(at), "v"(src), "s"(mma_scalar(lanes)) : "memory", "m0");
}
// four bytes per lane of `lanes` (lane l lands at lds_at + 4 l)
__device__ __forceinline__ void mma_copy4_lanes(const uint32_t* src, lds_u32* lds_at, uint64_t lanes) {
    const uint32_t at = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds_at)));
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %2\n\tglobal_load_lds_dword %1, off\n\ts_mov_b64 exec, -1"
                 : : "s"(at), "v"(src), "s"(mma_scalar(lanes)) : "memory", "m0");
}
template <int N> __device__ __forceinline__ void mma_wait() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
template <int N> __device__ __forceinline__ void mma_wait_n(uint32_t ahead) {   // at most N * ahead copies still in flight
    static_assert(3 * N <= 63, "vmcnt range");
    switch (ahead) {
    case 0: mma_wait<0>(); break;
    case 1: mma_wait<N>(); break;
    case 2: mma_wait<2 * N>(); break;
    default: mma_wait<3 * N>(); break;
    }
}

// Activation row served by operand-A slot i (the inverse of "row a -> result register a / 2 of half a % 2"); slots past the
// served rows repeat earlier rows (their results are never read).
template <int NAL> __device__ __forceinline__ uint32_t mma_slot_act(uint32_t i) {
    const uint32_t v = 4U * (i >> 3) + (i & 3U), h = (i >> 2) & 1U;
    return (2U * v + h) % mma_acts<NAL>();
}

// Per-lane byte offsets into a ring slot (constant over the sweep); matrix m's weights sit mma_weight_bytes m further on.
struct MmaLane {
    uint32_t head, fifth, quants, even, odd, table;
    bool sum_lane;
    uint32_t shift, even_slot;         // halves form: of the lane's sub-block in the header words; all ones where the lane's slot is of half 0
    uint32_t start;                    // Q6_K: the lane's row's first byte in its piece, of the first super-block; even_slot: all ones where the
                                       // lane's half of K is its slot's. Wide form: its slot's code sum of its half of the pair; even_slot: half 0
};

// Bit `bit` of every byte of a fifth-bit word, as bit 4 (Q5_K)
__device__ __forceinline__ u32x4 mma_fifth(const u32x4& qh, uint32_t bit) { return ((qh >> bit) & 0x01010101U) << 4; }

// One landed super-block: for each matrix the wavefront's two group dots of its 32 rows against every activation slot, then the
// lane's chain terms x[2P] + x[2P + 1] for its first nv activation rows. P is the wavefront's pair, a template argument so that
// the scale / min unpacking has constant shifts.
template <int FMT, int NAL, int NM, int P>
__device__ __forceinline__ void mma_stage_terms(const lds_u8* slot, const MmaLane& o, uint32_t nv, float (&term)[NM][NAL]) {
    typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
    typedef const __attribute__((address_space(3))) int32_t lds_i32;
    const u32x4 a_even = *(lds_u32x4*)(slot + o.even), a_odd = *(lds_u32x4*)(slot + o.odd);
    u32x4 hd[NM], q[NM], qh[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        hd[m] = *(lds_u32x4*)(slot + mma_weight_bytes<FMT>() * m + o.head);
        q[m] = *(lds_u32x4*)(slot + mma_weight_bytes<FMT>() * m + o.quants);
        if (FMT == kMmaQ5K) qh[m] = *(lds_u32x4*)(slot + mma_weight_bytes<FMT>() * m + o.fifth);
    }
    int32_t tab[NAL];
#pragma unroll
    for (int v = 0; v < NAL; ++v) tab[v] = *(lds_i32*)(slot + o.table + 128U * v);
    if (o.sum_lane) {                                       // quad lanes 2, 3 hold code sums: to float, once
#pragma unroll
        for (int v = 0; v < NAL; ++v) tab[v] = __builtin_bit_cast(int32_t, static_cast<float>(tab[v]));
    }
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        u32x4 lo = q[m] & 0x0f0f0f0fU, hi = (q[m] >> 4) & 0x0f0f0f0fU;
        if (FMT == kMmaQ5K) { lo |= mma_fifth(qh[m], 2 * P); hi |= mma_fifth(qh[m], 2 * P + 1); }
        const i32x16 zero = {0};
        const i32x16 dot_even = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a_even), __builtin_bit_cast(i32x4, lo), zero, 0, 0, 0);
        const i32x16 dot_odd = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a_odd), __builtin_bit_cast(i32x4, hi), zero, 0, 0, 0);
        uint32_t s0, m0, s1, m1;
        q4k_factors<2 * P>(hd[m], s0, m0);
        q4k_factors<2 * P + 1>(hd[m], s1, m1);
        const float d = half_bits_to_float(hd[m].x & 0xffffU), dm = half_bits_to_float(hd[m].x >> 16);
        const float D0 = d * static_cast<float>(s0), M0 = dm * static_cast<float>(m0);
        const float D1 = d * static_cast<float>(s1), M1 = dm * static_cast<float>(m1);
#pragma unroll
        for (int v = 0; v < NAL; ++v) {
            // the widest sweep skips the result registers past a short chunk, four at a time (straight-line code either way: a
            // loop exit here would turn the register arrays into indexed accesses)
            if (NAL > 8 && static_cast<uint32_t>(v & ~3) >= nv) continue;
            const float e0 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(tab[v], 0x00, 0xF, 0xF, true));
            const float e1 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(tab[v], 0x55, 0xF, 0xF, true));
            const float f0 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(tab[v], 0xAA, 0xF, 0xF, true));
            const float f1 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(tab[v], 0xFF, 0xF, 0xF, true));
            const float u0 = D0 * static_cast<float>(dot_even[v]), v0 = M0 * f0;
            const float u1 = D1 * static_cast<float>(dot_odd[v]), v1 = M1 * f1;
            const float x0 = e0 * (u0 - v0), x1 = e1 * (u1 - v1);
            term[m][v] = x0 + x1;
        }
    }
}

// The same in the wide form, one matrix a wavefront. v of a sub-block is an outer product (a minimum per weight row, a code sum per activation
// row), so a v_mfma_f32_32x32x2_f32 leaves it in the dots' layout: k = 0 carries sub-block 2p and k = 1 sub-block 2p + 1, each product
// with the other one's operands zero (a * b rounded once, + 0). A sub-block's terms take the place of its dots before the other's products
// are made, and the deltas come as broadcast reads, asked for in front of the products they wait with: 64 registers of results and deltas
// beside the accumulators, so that four wavefronts share a SIMD where two did (gate and up on one wavefront took 240). That is the bound of 128 registers a
// wavefront: the kernels spill 23 to 29 of gate / up and 4 to 7 of the down rows, written and read outside the stage loop, once a chunk or tile.
// Bound by the chain and by what a stage waits for (operands, products, the barrier), in about equal parts. Measured, before -> now: 1000 rows of
// hidden 2048 / ffn 768 / 128 experts gate / up 327 -> 297 us, down rows (16 activation rows a sweep before) 167 -> 146; dense 27648 x 5120,
// 32 rows gate / up 105 -> 95 us. Not faster: one wavefront for both matrices with u as one fma on biased dots, at two wavefronts a SIMD (a
// third fewer vector instructions, 301 us), the same without a barrier from rings of the wavefronts' own (305), a workgroup per chunk (307).
template <int FMT, int NAL>
__device__ __forceinline__ void mma_stage_wide(const lds_u8* slot, const MmaLane& o, uint32_t p, float (&acc)[NAL]) {
    typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
    typedef const __attribute__((address_space(3))) int32_t lds_i32;
    typedef float f32x16_t __attribute__((ext_vector_type(16)));
    const u32x4 hd = *(lds_u32x4*)(slot + o.head), q = *(lds_u32x4*)(slot + o.quants), a_even = *(lds_u32x4*)(slot + o.even);
    const int32_t sum = *(lds_i32*)(slot + o.start);
    u32x4 fifth = {0U, 0U, 0U, 0U};
    if (FMT == kMmaQ5K) fifth = *(lds_u32x4*)(slot + o.fifth);
    __builtin_amdgcn_sched_barrier(0);
    // (q4k_factors with the wavefront's shifts: six bits, or four and the two above another word's six)
    const bool high = p >= 2U;
    const uint32_t shift = 16U * (p & 1U), low_bits = high ? 4U : 6U, top_bits = high ? 2U : 0U;
    const uint32_t scales = high ? hd.w : hd.y, mins = high ? hd.w >> 4 : hd.z;
    const auto factor = [&](uint32_t word, uint32_t top, uint32_t at) {
        return static_cast<float>(__builtin_amdgcn_ubfe(word, at, low_bits) | (__builtin_amdgcn_ubfe(top, at + 6U, top_bits) << 4));
    };
    const float d = half_bits_to_float(hd.x & 0xffffU), dm = half_bits_to_float(hd.x >> 16);
    const float D0 = d * factor(scales, hd.y, shift), D1 = d * factor(scales, hd.y, shift + 8U);
    const float M = dm * factor(mins, hd.z, o.shift), f = static_cast<float>(sum);          // of the lane's half of the pair
    const auto products = [&](uint32_t odd, u32x4 n, const u32x4& a, i32x16& dot, f32x16_t& least) __attribute__((always_inline)) {
        if (FMT == kMmaQ5K) n |= mma_fifth(fifth, 2U * p + odd);
        const i32x16 zero = {0};
        const f32x16_t none = {0.0F};
        const uint32_t in = odd ? ~o.even_slot : o.even_slot;
        dot = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, n), zero, 0, 0, 0);
        least = __builtin_amdgcn_mfma_f32_32x32x2f32(f_of(b_of(f) & in), f_of(b_of(M) & in), none, 0, 0, 0);
    };
    i32x16 dot;
    f32x16_t least;
    products(0, q & 0x0f0f0f0fU, a_even, dot, least);
    __builtin_amdgcn_sched_barrier(0);
    const u32x4 a_odd = *(lds_u32x4*)(slot + o.odd);
    float e[NAL], x0[NAL];
#pragma unroll
    for (int v = 0; v < NAL; ++v) e[v] = *(const lds_f32*)(slot + o.table + 128U * v);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < NAL; ++v) x0[v] = e[v] * (D0 * static_cast<float>(dot[v]) - least[v]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < NAL; ++v) e[v] = *(const lds_f32*)(slot + o.table + 128U * v + 4U);
    products(1, (q >> 4) & 0x0f0f0f0fU, a_odd, dot, least);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < NAL; ++v) acc[v] = acc[v] + (x0[v] + e[v] * (D1 * static_cast<float>(dot[v]) - least[v]));
    __builtin_amdgcn_sched_barrier(0);
}

// The same for few activation rows (NAL == 2), where the scales, the nibbles and the layout's own moves outweigh the chain: each half of
// the wavefront takes ONE of the pair's sub-blocks, for every activation row. Slot i serves activation row v = 4 (i / 8) + i % 4 in half
// (i / 4) % 2, and its codes are of sub-block 2p in the slots of half 0, of 2p + 1 in those of half 1; two products - each with the other
// half's slots zeroed - accumulate into one result, whose register v holds activation row v's dot with sub-block 2p in the lanes of half 0
// and with sub-block 2p + 1 in those of half 1. A lane then decodes one scale and one minimum instead of two, and the terms of two
// activation rows meet through one exchange of the halves: x[2p] + x[2p + 1] of row 2v + h lands where the wide form leaves it.
// (4 activation rows, gate and up: 140 -> 115 vector instructions a stage; dense 27648 x 5120, 4 rows 76.1 -> 75.0 us. With 8 activation rows, as many conversions and two products in a row, it is the slower one: 100 rows of
// hidden 2048 / ffn 768 / 128 experts 162.0 against 160.2 us, 90 rows of hidden 4096 / ffn 1536 / 64 experts 326 against 321.)
template <int FMT, int NAL, int NM, bool HIGH>
__device__ __forceinline__ void mma_stage_terms_halves(const lds_u8* slot, const MmaLane& o, uint32_t p, float (&term)[NM][NAL]) {
    typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
    typedef const __attribute__((address_space(3))) int32_t lds_i32;
    const u32x4 codes = *(lds_u32x4*)(slot + o.even);
    u32x4 hd[NM], q[NM], qh[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        hd[m] = *(lds_u32x4*)(slot + mma_weight_bytes<FMT>() * m + o.head);
        q[m] = *(lds_u32x4*)(slot + mma_weight_bytes<FMT>() * m + o.quants);
        if (FMT == kMmaQ5K) qh[m] = *(lds_u32x4*)(slot + mma_weight_bytes<FMT>() * m + o.fifth);
    }
    float e[2 * NAL], f[2 * NAL];
#pragma unroll
    for (int a = 0; a < 2 * NAL; ++a) {
        e[a] = *(const lds_f32*)(slot + o.table + 64U * a);
        f[a] = static_cast<float>(*(lds_i32*)(slot + o.table + 64U * a + 32U));
    }
    const u32x4 a_even = codes & o.even_slot, a_odd = codes & ~o.even_slot;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        u32x4 lo = q[m] & 0x0f0f0f0fU, hi = (q[m] >> 4) & 0x0f0f0f0fU;
        if (FMT == kMmaQ5K) { lo |= mma_fifth(qh[m], 2U * p); hi |= mma_fifth(qh[m], 2U * p + 1U); }
        const i32x16 zero = {0};
        i32x16 dot = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a_even), __builtin_bit_cast(i32x4, lo), zero, 0, 0, 0);
        dot = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a_odd), __builtin_bit_cast(i32x4, hi), dot, 0, 0, 0);
        uint32_t sc, mn;                                       // (q4k_factors with the shift of the lane's sub-block)
        if (!HIGH) {
            sc = __builtin_amdgcn_ubfe(hd[m].y, o.shift, 6U);
            mn = __builtin_amdgcn_ubfe(hd[m].z, o.shift, 6U);
        } else {
            sc = __builtin_amdgcn_ubfe(hd[m].w, o.shift, 4U) | (__builtin_amdgcn_ubfe(hd[m].y, o.shift + 6U, 2U) << 4);
            mn = __builtin_amdgcn_ubfe(hd[m].w, o.shift + 4U, 4U) | (__builtin_amdgcn_ubfe(hd[m].z, o.shift + 6U, 2U) << 4);
        }
        const float D = half_bits_to_float(hd[m].x & 0xffffU) * static_cast<float>(sc), M = half_bits_to_float(hd[m].x >> 16) * static_cast<float>(mn);
#pragma unroll
        for (int v = 0; v < NAL; ++v) {
            const float u0 = D * static_cast<float>(dot[2 * v]), v0 = M * f[2 * v], x0 = e[2 * v] * (u0 - v0);
            const float u1 = D * static_cast<float>(dot[2 * v + 1]), v1 = M * f[2 * v + 1], x1 = e[2 * v + 1] * (u1 - v1);
            const auto met = __builtin_amdgcn_permlane32_swap(b_of(x0), b_of(x1), false, false);      // (half 0's rows 2v, half 1's rows 2v + 1)
            term[m][v] = f_of(met[0]) + f_of(met[1]);
        }
    }
}
template <int NAL> constexpr bool mma_halves() { return NAL == 2; }

// N words of LDS from a 2-byte aligned place
template <int N> __device__ __forceinline__ void mma_words(const lds_u8* at, uint32_t (&out)[N]) {
    typedef const __attribute__((address_space(3))) uint32_t lds_word;
    const uint32_t address = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(at)), shift = address & 3U;
    lds_word* const aligned = (lds_word*)(uintptr_t)(address & ~3U);
    uint32_t raw[N + 1];
#pragma unroll
    for (int i = 0; i <= N; ++i) raw[i] = aligned[i];           // (the word behind an aligned run lies inside the slot: read, unused)
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = __builtin_amdgcn_alignbyte(raw[i + 1], raw[i], shift);
}

// One landed stage of down rows in the other formats of the reference (256 weights of every row), added to the wavefront's accumulators.
// Same products and result layout as above.
//   Q8_0, Q5_1: wavefront p is chain p, which owns groups p and p + 4 of the stage, each added by itself (down_groups.hpp):
//     first = d * float(dot); Q5_1: combined = first + m * float(code sum); chain += delta * combined.
//   Q6_K: wavefront p is pair p (groups 2p, 2p + 1; q6k_quads.hpp): integer = s0 * dot(first 16) + s1 * dot(last 16),
//     term = delta * (d * float(integer)), acc += term_2p + term_(2p+1). One product of K = 32 gives both dots: result register 2v + s of a
//     lane belongs to activation row 2v + h and the group's half s, because slot i carries the codes of its half of K only (zeros in the
//     other) - so 16 activation rows at most.
// stage: of the row; where in its piece a Q6_K row's block starts (two bytes further every super-block: 210 = 13 * 16 + 2).
template <int FMT, int NAL>
__device__ __forceinline__ void mma_stage_other(const lds_u8* slot, const MmaLane& o, uint32_t p, uint32_t stage, float (&acc)[NAL]) {
    typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
    typedef const __attribute__((address_space(3))) int32_t lds_i32;
    typedef const __attribute__((address_space(3))) uint16_t lds_u16;
    static_assert(NAL <= 8, "sixteen result registers");
    u32x4 a0 = *(lds_u32x4*)(slot + o.even), a1 = *(lds_u32x4*)(slot + o.odd);
    int32_t tab[NAL];
#pragma unroll
    for (int v = 0; v < NAL; ++v) tab[v] = *(lds_i32*)(slot + o.table + 128U * v);
    if (FMT == kMmaQ51 && o.sum_lane) {
#pragma unroll
        for (int v = 0; v < NAL; ++v) tab[v] = __builtin_bit_cast(int32_t, static_cast<float>(tab[v]));
    }
    uint32_t q0[4], q1[4];
    float d0, d1 = 0.0F, m0 = 0.0F, m1 = 0.0F;
    int s[2][2] = {{0, 0}, {0, 0}};
    if constexpr (FMT == kMmaQ80) {
        const lds_u8* const b0 = slot + o.quants;
        mma_words<4>(b0 + o.fifth, q0);
        mma_words<4>(b0 + 136U + o.fifth, q1);
        d0 = half_bits_to_float(*(lds_u16*)b0);
        d1 = half_bits_to_float(*(lds_u16*)(b0 + 136U));
    } else if constexpr (FMT == kMmaQ51) {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        typedef const __attribute__((address_space(3))) u32x2 lds_u32x2;
        const lds_u8* const b0 = slot + o.quants;
        uint32_t fifth[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const u32x2 head = *(lds_u32x2*)(b0 + 96 * k), n0 = *(lds_u32x2*)(b0 + 96 * k + 8), n1 = *(lds_u32x2*)(b0 + 96 * k + 16);
            uint32_t (&q)[4] = k ? q1 : q0;
            const uint32_t n[4] = {n0.x, n0.y, n1.x, n1.y};
            fifth[k] = head.y >> (4U * o.shift);                     // o.shift: 4 in half 1 (weights 16 .. 31: high nibbles, bits 16 ..)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                q[i] = ((n[i] >> o.shift) & 0x0f0f0f0fU) | ((((fifth[k] >> (4 * i)) & 15U) * 0x00204081U & 0x01010101U) << 4);
            (k ? d1 : d0) = half_bits_to_float(head.x & 0xffffU);
            (k ? m1 : m0) = half_bits_to_float(head.x >> 16);
        }
    } else {
        const lds_u8* const block = slot + o.head + ((o.start + 2U * stage) & 15U);
        uint32_t qh[4], t[1];
        mma_words<4>(block + o.quants, q0);
        mma_words<4>(block + o.quants + 32U, q1);
        mma_words<4>(block + o.fifth, qh);
        mma_words<1>(block + 192U + 4U * p, t);
        d0 = half_bits_to_float(*(lds_u16*)(block + 208U)) * 0.25F;
        // four times the weight, ((nibble | pair << 4) - 32) << 2, is the six bits at the top of the byte with the highest one flipped; the
        // factor leaves with d (exact: a power of two)
        const uint32_t nibbles = p & 1U ? 2U : 30U, pairs = p & 1U ? 30U : 26U;             // rotations to the right
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t n0 = __builtin_amdgcn_alignbit(q0[i], q0[i], nibbles), n1 = __builtin_amdgcn_alignbit(q1[i], q1[i], nibbles);
            const uint32_t h0 = __builtin_amdgcn_alignbit(qh[i], qh[i], pairs), h1 = __builtin_amdgcn_alignbit(qh[i], qh[i], pairs + 2U);
            q0[i] = ((n0 & 0x3c3c3c3cU) | (h0 & 0xc0c0c0c0U)) ^ 0x80808080U;
            q1[i] = ((n1 & 0x3c3c3c3cU) | (h1 & 0xc0c0c0c0U)) ^ 0x80808080U;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i >> 1][i & 1] = static_cast<int8_t>(t[0] >> (8 * i));
        a0 = a0 & o.even_slot;
        a1 = a1 & o.even_slot;
    }
    const u32x4 w0 = {q0[0], q0[1], q0[2], q0[3]}, w1 = {q1[0], q1[1], q1[2], q1[3]};
    const i32x16 zero = {0};
    const i32x16 dot0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a0), __builtin_bit_cast(i32x4, w0), zero, 0, 0, 0);
    const i32x16 dot1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a1), __builtin_bit_cast(i32x4, w1), zero, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < NAL; ++v) {
        const float e0 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(tab[v], 0x00, 0xF, 0xF, true));
        const float e1 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(tab[v], 0x55, 0xF, 0xF, true));
        if constexpr (FMT == kMmaQ6K) {
            const int i0 = __mul24(s[0][0], dot0[2 * v]) + __mul24(s[0][1], dot0[2 * v + 1]);
            const int i1 = __mul24(s[1][0], dot1[2 * v]) + __mul24(s[1][1], dot1[2 * v + 1]);
            const float t0 = e0 * (d0 * static_cast<float>(i0)), t1 = e1 * (d0 * static_cast<float>(i1));
            acc[v] = acc[v] + (t0 + t1);
        } else {
            float c0 = d0 * static_cast<float>(dot0[v]), c1 = d1 * static_cast<float>(dot1[v]);
            if constexpr (FMT == kMmaQ51) {
                const float f0 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(tab[v], 0xAA, 0xF, 0xF, true));
                const float f1 = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(tab[v], 0xFF, 0xF, 0xF, true));
                c0 = c0 + (m0 * f0);
                c1 = c1 + (m1 * f1);
            }
            acc[v] = acc[v] + (e0 * c0);
            acc[v] = acc[v] + (e1 * c1);
        }
    }
}
// The activation rows of a run and where their results go, resolved once by one wavefront: addresses of the A8 image of row a (codes,
// deltas, sums), OUT more addresses for the emitter, and the row's assignment.
template <int NAL, int OUT> constexpr uint32_t mma_row_words() { return (3U + OUT) * mma_acts<NAL>(); }

// A run of `tiles` 32-row tiles, back to back in memory (NM matrices' tiles share the activation rows), of `stages` super-blocks against
// nacts <= 2 NAL activation rows. Wavefront p keeps pair accumulator p of (row j, activation row 2v + h) in acc[m][v]; at the end of a tile
// value = (acc0 + acc1) + (acc2 + acc3) over the four wavefronts, through `red`: wavefront w receives the values of result registers
// v = w, w + 4, ... and hands (tile, v, its lane, values of the NM matrices) to emit.
//   rows.word(a): address of a word that names activation row a (its place in the plan's order); rows.put(a, nacts, word): leaves the row's
//   addresses in rows.at. Wavefront 3 asks for the words first, then every wavefront starts the weights of the first stages, so the
//   look-up is in flight beside them. Rows::kDirect: the addresses need no look-up (rows.codes / rows.table), every wavefront works its
//   own out and starts whole stages (but for four rows), so the first product waits for the first stage only; the row table serves the
//   emitter, or (no kPut) nobody.
//   WIDE: mma_stage_wide's form, four wavefronts for each of the NM matrices. tile_rows: rows from a tile to the next.
//   RUNS: several tiles (else one: none of a run's bookkeeping; gate and up of a dense block, 27648 x 5120, 8 rows: 32.4 -> 31.9 us, and 33.4 with
//   the weights of both first stages in front of the codes and the row table written in front of the first product).
//
// TEAMS > 1 (a matrix of few, long rows gives few workgroups, each with K / 256 dependent stages; one tile a run): TEAMS x 4 wavefronts;
// team t takes super-blocks t, TEAMS + t, ... of the same 32 rows, so TEAMS stages are in the pipes at once. The chain order is
// kept by team 0, which adds the terms of every super-block in ascending order: its own from registers, the other teams'
// from an LDS exchange buffer, one stage group behind (the group's barrier publishes them).
// Every wavefront of the workgroup calls this; ring, row table and `red` are free again when it returns.
template <int FMT, int NAL, int DEPTH, int TEAMS, int NM, bool RUNS, bool WIDE, class Rows, class Emit>
__device__ __forceinline__ void mma_run(lds_u8* ring, lds_f32* xbuf, lds_f32* red, const uint8_t* const (&wrows)[NM], size_t row_stride, uint32_t stages,
                                        uint32_t tiles, uint32_t tile_rows, uint32_t nacts, Rows rows, Emit emit) {
    constexpr uint32_t ACTS = mma_acts<NAL>(), CC = mma_code_copies<NAL>(), TOTAL = mma_copies<FMT, NAL, NM>(), SLOT = mma_slot_bytes<FMT, NAL, NM>();
    constexpr uint32_t CW = mma_weight_copies<FMT>(), PIECES = mma_pieces<FMT>(), PITCH = mma_pitch<FMT>(), BYTES = mma_block_bytes<FMT>();
    // In the ring every wavefront issues PERW copies a stage - past the last one it copies the last one's first piece again, the same bytes to
    // the same place - so there are no branches on the wavefront's number and one count to wait for. The run's first stages are issued in
    // two parts of as many copies as a wavefront has there, and awaited whole.
    constexpr uint32_t W = mma_waves<NM, WIDE>(), MATS = 4U * NM / W;                             // wavefronts of a team; matrices of a wavefront
    constexpr uint32_t PERW = (TOTAL + W - 1U) / W, WEIGHTS = CW * NM, WEIGHTS_LAST = (WEIGHTS - 3U + W - 1U) / W;        // (weight copies of wavefront 3)
    constexpr uint32_t XTEAM = 4U * NAL * 64U;                                                  // floats one team exchanges per group
    static_assert(DEPTH >= 2 && DEPTH <= 4, "ring depth");
    static_assert(TEAMS == 1 || (NM == 1 && NAL <= 8 && FMT == kMmaQ4K), "stage teams serve one matrix, every result register");
    static_assert(!WIDE || (TEAMS == 1 && (FMT == kMmaQ4K || FMT == kMmaQ5K)), "wide form");
    static_assert(NM == 1 || FMT == kMmaQ4K || FMT == kMmaQ5K, "gate and up rows");
    static_assert(CW >= 4U && PIECES >= 8U, "copies 0 .. 3 are of whole waves");
    const uint32_t lane = threadIdx.x & 63U, j = lane & 31U, h = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = wave % W, p = w & 3U, matrix = w >> 2, team = wave / W;
    const uint32_t groups = (stages + TEAMS - 1U) / TEAMS;                                     // of a tile
    const uint32_t my_groups = team < stages - (groups - 1U) * TEAMS ? groups : groups - 1U;   // groups in which this team has a super-block
    const uint32_t total = RUNS ? groups * tiles : groups, my_total = TEAMS == 1 ? total : my_groups;
    const uint32_t nv = (nacts + 1U) / 2U;

    // ---- this wavefront's copies of a stage, copy c = 4k + p: CW per matrix (the pieces of 16 bytes of a row, rows PITCH apart; the
    // last moves half a kilobyte), codes (16 pieces per row, piece t at position (t + a) % 16), table (per row [8 deltas][8 sums])
    const uint8_t* src[PERW];
    uint32_t step[PERW], lands[PERW], piece_at[PERW];
    uint64_t lanes[PERW];
#pragma unroll
    for (uint32_t k = 0; k < PERW; ++k) {
        const uint32_t c = W * k + w;
        if (c < WEIGHTS) {
            const uint32_t m = c / CW, i = c - CW * m, s = 64U * i + lane < kMmaRows * PITCH ? 64U * i + lane : 0U, r = s / PITCH;
            const uint32_t piece = s - PITCH * r < PIECES ? s - PITCH * r : PIECES - 1U;
            src[k] = wrows[m < NM ? m : 0] + static_cast<size_t>(r) * row_stride + BYTES * team;
            if (FMT == kMmaQ6K) piece_at[k] = 16U * piece;           // (from the piece that the row's block starts in, found when it is copied)
            else src[k] += 16U * piece;
            step[k] = BYTES * TEAMS;
            lands[k] = mma_weight_bytes<FMT>() * m + 1024U * i;
            lanes[k] = i == CW - 1U ? 0xffffffffULL : ~0ULL;
        } else if (c < WEIGHTS + CC) {
            src[k] = nullptr;
            step[k] = 256U * TEAMS;
            lands[k] = mma_codes_at<FMT, NM>() + 1024U * (c - WEIGHTS);
            lanes[k] = ~0ULL;
        } else {
            src[k] = nullptr;
            step[k] = 32U * TEAMS;
            lands[k] = mma_table_at<FMT, NAL, NM>() + 1024U * ((c < TOTAL ? c : TOTAL - 1U) - WEIGHTS - CC);
            lanes[k] = c >= TOTAL ? 1ULL : ACTS >= 16U ? ~0ULL : (1ULL << (4U * ACTS)) - 1ULL;
        }
    }
    // The first stages in one part each, or the weights of both first (27648 x 5120, 4 rows 63.0 | 62.7 us, 8 rows 69.0 | 71.1; 14848 x 5120, 44 rows
    // 141.4 | 143.5: with more rows a stage's codes are as many bytes as its weights).
    constexpr bool WHOLE = Rows::kDirect && (!Rows::kPut || NAL > 2);
    const size_t next_tile = tile_rows * row_stride - BYTES * static_cast<size_t>(stages);       // from a tile's end to the next one's start
    uint32_t issued = 0, issue_stage = 0;
    // copies of the next stage into a slot; PART 1: the weights (of the run's first stages, whose activation rows are not known yet), 2: the rest
    const auto start = [&](auto part_constant, lds_u8* slot) __attribute__((always_inline)) {
        constexpr int part = decltype(part_constant)::value;
#pragma unroll
        for (uint32_t k = 0; k < PERW; ++k) {
            if (part != 0 && (W * k + w < WEIGHTS) != (part == 1)) continue;
            const uint8_t* from = src[k];
            if (FMT == kMmaQ6K && W * k + w < WEIGHTS) from = reinterpret_cast<const uint8_t*>(reinterpret_cast<uintptr_t>(from) & ~static_cast<uintptr_t>(15)) + piece_at[k];
            if (W == 4U && part == 0 && k == 0U) mma_copy16(from, slot + lands[k]);            // (copies 0 .. 3: weights of a whole wave)
            else mma_copy16_lanes(from, slot + lands[k], lanes[k]);
            src[k] += step[k];
        }
        if (RUNS && ++issue_stage == stages) {
            issue_stage = 0;
#pragma unroll
            for (uint32_t k = 0; k < PERW; ++k) {
                const bool weights = W * k + w < WEIGHTS;
                if (part == 0 || weights == (part == 1)) src[k] += weights ? next_tile : 0U - static_cast<size_t>(step[k]) * stages;
            }
        }
    };
    const auto slot_of = [&](uint32_t s) { return ring + SLOT * (s * TEAMS + team); };
    const uint32_t first = my_total < DEPTH - 1U ? my_total : DEPTH - 1U;
    const auto start_weights = [&]() {
        for (uint32_t s = 0; s < first; ++s) start(std::integral_constant<int, 1>{}, slot_of(s));
    };
    const auto row_of_codes = [&](uint32_t k) { return (64U * (W * k + w - WEIGHTS) + lane) >> 4; };                            // of the lane's 16 bytes
    const auto row_of_table = [&](uint32_t k) {
        const uint32_t c = W * k + w < TOTAL ? W * k + w : TOTAL - 1U;
        return (16U * (c - WEIGHTS - CC) + (lane >> 2)) % ACTS;
    };
    const auto set_rows = [&](auto codes_of, auto table_of) {
#pragma unroll
        for (uint32_t k = 0; k < PERW; ++k) {
            const uint32_t c = W * k + w;
            if (c >= WEIGHTS && c < WEIGHTS + CC) {
                const uint32_t a = row_of_codes(k);
                src[k] = codes_of(a) + 16U * (((lane & 15U) - a) & 15U) + 256U * team;
            } else if (c >= WEIGHTS + CC) {
                const uint32_t q = lane & 3U;
                src[k] = table_of(row_of_table(k), q < 2U) + 16U * (q & 1U) + 32U * team;
            }
        }
    };
    if constexpr (Rows::kDirect) {
        if (!WHOLE) start_weights();
        set_rows([&](uint32_t a) { return rows.codes(a < nacts ? a : 0U); }, [&](uint32_t a, bool deltas) { return rows.table(a < nacts ? a : 0U, deltas); });
    } else {
        if (wave == 3U) {
            // (the words land in LDS like everything else: a register that a load in flight writes could be copied before it does)
            mma_copy4_lanes(rows.word(lane < nacts ? lane : 0U), rows.slot, (1ULL << ACTS) - 1ULL);
            start_weights();
            if (DEPTH > 2 && first == DEPTH - 1U) mma_wait<WEIGHTS_LAST * (DEPTH - 1)>();
            else mma_wait<WEIGHTS_LAST>();
            if (lane < ACTS) rows.put(lane, nacts, rows.slot[lane]);
        } else start_weights();
        mma_barrier();
        set_rows([&](uint32_t a) { return reinterpret_cast<const uint8_t*>(rows.at[a]); },
                 [&](uint32_t a, bool deltas) { return reinterpret_cast<const uint8_t*>(rows.at[(deltas ? Rows::kActs : 2U * Rows::kActs) + a]); });
    }

    MmaLane o;
    {
        const uint32_t ai = mma_slot_act<NAL>(j), c_base = mma_codes_at<FMT, NM>() + 256U * ai;
        o.head = 16U * PITCH * j;
        if (FMT == kMmaQ4K || FMT == kMmaQ5K) {
            o.fifth = 16U * PITCH * j + 16U + 16U * h;
            o.quants = 16U * PITCH * j + (FMT == kMmaQ5K ? 48U : 16U) + 32U * p + 16U * h;
        } else if (FMT == kMmaQ6K) {                              // from the block's first byte: nibbles, bit pairs
            o.quants = 64U * (p >> 1) + 16U * h;
            o.fifth = 128U + 32U * (p >> 1) + 16U * h;
            o.start = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(wrows[0]) + j * row_stride) & 15U;
        } else {                                                  // chain p: block p of the stage, codes 16 h ..
            o.quants = 16U * PITCH * j + (FMT == kMmaQ80 ? 34U : 24U) * p;
            o.fifth = 2U + 16U * h;
            o.shift = 4U * h;
        }
        // the lane's activation slot: groups 2p and 2p + 1, of chain p groups p and p + 4 (16-byte pieces 2 g + h of its row)
        constexpr bool CHAINS = FMT == kMmaQ80 || FMT == kMmaQ51;
        const uint32_t g0 = CHAINS ? p : 2U * p, g1 = CHAINS ? p + 4U : 2U * p + 1U;
        o.even = c_base + 16U * ((2U * g0 + h + ai) & 15U);
        o.odd = c_base + 16U * ((2U * g1 + h + ai) & 15U);
        if (FMT == kMmaQ6K) {                                     // result register 2v + s: activation row 2v + h, half s of the group
            const uint32_t reg = 4U * (j >> 3) + (j & 3U), act = ((reg & ~1U) + ((j >> 2) & 1U)) & (ACTS - 1U), base = mma_codes_at<FMT, NM>() + 256U * act;
            o.even = base + 16U * ((2U * g0 + h + act) & 15U);
            o.odd = base + 16U * ((2U * g1 + h + act) & 15U);
            o.even_slot = (reg & 1U) == h ? ~0U : 0U;
        }
        // quad lane 0, 1: the deltas of g0, g1; quad lane 2, 3: their code sums
        o.table = mma_table_at<FMT, NAL, NM>() + 64U * h + 4U * ((lane & 1U ? g1 : g0) + 4U * (lane & 2U));
        o.sum_lane = (lane & 2U) != 0;
        if constexpr (WIDE) {
            o.head += mma_weight_bytes<FMT>() * matrix;
            o.fifth += mma_weight_bytes<FMT>() * matrix;
            o.quants += mma_weight_bytes<FMT>() * matrix;
            o.table = mma_table_at<FMT, NAL, NM>() + 64U * h + 8U * p;                          // the deltas of activation row 2v + h
            o.start = mma_table_at<FMT, NAL, NM>() + 64U * ai + 32U + 4U * (2U * p + h);        // the code sum of the lane's slot and half of the pair
            o.shift = 16U * (p & 1U) + 8U * h;
            o.even_slot = h ? 0U : ~0U;
        }
        if constexpr (!WIDE && mma_halves<NAL>() && (FMT == kMmaQ4K || FMT == kMmaQ5K)) {
            const uint32_t odd = (j >> 2) & 1U, act = (4U * (j >> 3) + (j & 3U)) & (ACTS - 1U);
            o.even = mma_codes_at<FMT, NM>() + 256U * act + 16U * ((4U * p + 2U * odd + h + act) & 15U);
            o.table = mma_table_at<FMT, NAL, NM>() + 4U * (2U * p + h);
            o.shift = 16U * (p & 1U) + 8U * h;
            o.even_slot = odd ? 0U : ~0U;
        }
    }

    float acc[MATS][NAL], own[NAL];
#pragma unroll
    for (int v = 0; v < NAL; ++v) own[v] = 0.0F;
    const auto clear = [&]() {
#pragma unroll
        for (uint32_t m = 0; m < MATS; ++m)
#pragma unroll
            for (int v = 0; v < NAL; ++v) acc[m][v] = 0.0F;
    };
    clear();
    // team 0: the terms of group g (its own, then teams 1 .. of the super-blocks that exist), in super-block order
    const auto fold = [&](uint32_t g) {
#pragma unroll
        for (int v = 0; v < NAL; ++v) acc[0][v] = acc[0][v] + own[v];
#pragma unroll
        for (uint32_t t = 1; t < TEAMS; ++t) {
            if (g * TEAMS + t < stages) {
                const lds_f32* x = xbuf + ((g & 1U) * (TEAMS - 1U) + (t - 1U)) * XTEAM + p * NAL * 64U + lane;
#pragma unroll
                for (int v = 0; v < NAL; ++v) acc[0][v] = acc[0][v] + x[v * 64];
            }
        }
    };
    const auto leave = [&]() {
#pragma unroll
        for (uint32_t m = 0; m < MATS; ++m)
#pragma unroll
            for (int v = 0; v < NAL; ++v) red[((m * 4U + w) * NAL + v) * 64U + lane] = acc[m][v];
    };
    const auto emit_tile = [&](uint32_t tile) {
        uint32_t lane = threadIdx.x & 63U;
        asm volatile("" : "+v"(lane));         // (what follows from it is worked out here, once a tile, not held in registers over the sweep)
        for (uint32_t v = w; v < nv; v += W) {
            float value[NM];
#pragma unroll
            for (uint32_t m = 0; m < NM; ++m) {
                const lds_f32* x = red + (m * 4U * NAL + v) * 64U + lane;
                const float left = x[0] + x[NAL * 64U], right = x[2U * NAL * 64U] + x[3U * NAL * 64U];
                value[m] = left + right;
            }
            emit(tile, v, lane, value);
        }
    };

    // ---- the ring of stage groups
    issue_stage = 0;
    for (; issued < first; ++issued) start(std::integral_constant<int, WHOLE ? 0 : 2>{}, slot_of(issued));
    if (Rows::kDirect && Rows::kPut && wave == 3U && lane < ACTS) rows.put(lane, nacts, 0U);       // (first read behind the first stage's barrier)
    uint32_t issue_slot = DEPTH - 1U, compute_slot = 0, stage = 0, tile = 0;
    const auto issue = [&]() {
        if (issued < my_total) { start(std::integral_constant<int, 0>{}, slot_of(issue_slot)); ++issued; }
        issue_slot = issue_slot + 1U == DEPTH ? 0U : issue_slot + 1U;
    };
    for (uint32_t g = 0; g < total; ++g) {
        // this wavefront's stages started after its stage of group g (first stages in two parts are not PERW copies each: all of them before the first)
        if (g < my_total) mma_wait_n<PERW>(!WHOLE && g == 0U ? 0U : issued - 1U - g);
        mma_barrier();         // every copy of group g is in, the slots of group g - 1 are free, its exchanged terms are written
        // The values of the tile before leave in its successor's first stage. They are stores, which the counted waits count too: before
        // the stage's copies they delay those a little, behind them the next wait would wait for copies that it does not need -
        // except in a ring of two slots, whose every wait is for everything.
        if (DEPTH == 2) issue();
        if (RUNS && stage == 0U && g != 0U) {
            emit_tile(tile - 1U);
            if (stages == 1U) mma_barrier();                     // (the next values are written in this stage)
        }
        if (DEPTH != 2) issue();
        if (TEAMS > 1 && team == 0U && g > 0U) fold(g - 1U);
        if (g < my_total) {
            const lds_u8* slot = ring + SLOT * (compute_slot * TEAMS + team);
            float term[MATS][NAL];
            if constexpr (WIDE) mma_stage_wide<FMT, NAL>(slot, o, p, acc[0]);
            else if constexpr (FMT != kMmaQ4K && FMT != kMmaQ5K) mma_stage_other<FMT, NAL>(slot, o, p, RUNS ? stage : g, acc[0]);
            else if constexpr (mma_halves<NAL>()) {
                if (p < 2U) mma_stage_terms_halves<FMT, NAL, NM, false>(slot, o, p, term);
                else mma_stage_terms_halves<FMT, NAL, NM, true>(slot, o, p, term);
            } else switch (p) {
            case 0: mma_stage_terms<FMT, NAL, NM, 0>(slot, o, nv, term); break;
            case 1: mma_stage_terms<FMT, NAL, NM, 1>(slot, o, nv, term); break;
            case 2: mma_stage_terms<FMT, NAL, NM, 2>(slot, o, nv, term); break;
            default: mma_stage_terms<FMT, NAL, NM, 3>(slot, o, nv, term); break;
            }
            if ((FMT != kMmaQ4K && FMT != kMmaQ5K) || WIDE) {
            } else if (TEAMS == 1) {
#pragma unroll
                for (uint32_t m = 0; m < MATS; ++m)
#pragma unroll
                    for (int v = 0; v < NAL; ++v) {
                        if (NAL > 8 && static_cast<uint32_t>(v & ~3) >= nv) continue;
                        acc[m][v] = acc[m][v] + term[m][v];
                    }
            } else if (team == 0U) {
#pragma unroll
                for (int v = 0; v < NAL; ++v) own[v] = term[0][v];
            } else {
                lds_f32* x = xbuf + ((g & 1U) * (TEAMS - 1U) + (team - 1U)) * XTEAM + p * NAL * 64U + lane;
#pragma unroll
                for (int v = 0; v < NAL; ++v) x[v * 64] = term[0][v];
            }
        }
        compute_slot = compute_slot + 1U == DEPTH ? 0U : compute_slot + 1U;
        if (RUNS && ++stage == stages) {
            stage = 0;
            ++tile;
            leave();
            clear();
        }
    }
    if (RUNS || TEAMS > 1) mma_barrier();      // the last values (TEAMS > 1: the last exchanged terms) are written; no copy is in flight
    if (!RUNS) {
        if (team == 0U) {
            if (TEAMS > 1) fold(groups - 1U);
            leave();
        }
        mma_barrier();
        if (team == 0U) emit_tile(0U);
    } else emit_tile(tiles - 1U);
    mma_barrier();             // every LDS read is done
}

}  // namespace strix950
