// Prefill form of the routed experts for gfx950: an expert-grouped GEMM on the fp16 matrix cores, Q4_K, Q5_K or Q8_0 tensors. Every wave
// expands its own weight rows into MFMA operands in registers (no weight passes through LDS) and multiplies them with 32-token tiles read
// from LDS. This is the path's second arithmetic class (the reference's FAST forms, include/strix/cuda/qwen_moe.hpp:100-101
// "bit-changing"); its parity target is the exact-weight product (include/strix/ds41_layer.hpp:96-121) within the stated tolerance, not the
// integer-dot class's bits: no weight is rounded.
//
// Arithmetic, Q4_K. w = d_b (sc_j q) - dmin_b m_j (src/ggml_dequant.cpp:119-130). The MFMA operand of a weight is the fp16 number
// 2^-14 sc_j q, made by ONE packed multiplication per two weights (SCALED below; sc q <= 945: exact). With S_bj[t] = sum of x_k[t]
// over sub-block j of super-block b,
//   out[t][f] = sum_b (2^14 d_b[f] P_b[t][f] - dmin_b[f] L_b[t][f]),
//   P_b = sum_(k in b) 2^-14 sc_j q_k x_k[t],   L_b = sum_(j in b) m_j S_bj[t]   (fp16 MFMAs, fp32 accumulation),
// S as fp16 hi + lo in one product (K = 8 + 8) against the exact integers m_j. In the down product the activation h is carried as
// fp16 hi + lo as well, so that the only roundings of the whole expert are fp32 accumulations. Before, the operand was 1024 + sc q and
// 1024 d + dmin m a second operand split into hi + lo: 64 | 333 rows of hidden 2048 / ffn 768 / 128 experts 96.4 | 163.3 us, now 90.8 | 151.0 (with
// a super-block's quants from one address), 300 rows of hidden 5120 / ffn 1536 / 160 experts 874 -> 811, Q5_K, 333 rows 192 -> 178;
// with four token tiles 1000 rows 266 -> 260. Error against 64 bits 1.9e-6 -> 5.5e-7, Q5_K 7.4e-8 -> 6.2e-8.
// Q5_K: the same blocks with 32 fifth-bit bytes after the factors (bit j of byte k for element k of sub-block j). sc q <= 1953 is an exact
// fp16 integer: fma(1024 + q, sc, -1024 sc), packed; no 2^14.
// Q8_0: one d per 32 codes and no minimum (src/ggml_dequant.cpp:84-87): the codes are exact fp16 integers, (1152 + code) - 1152, P is of a block.
//
// Work decomposition. A plan item holds at most 128 rows of one expert. A 512-thread workgroup owns (item, 256 weight rows):
// 128 gate + 128 up rows (MODE 0) or 256 down rows (MODE 1). Wave w owns 32 of the rows x all 128 tokens: accumulators
// 4 token tiles x 16 registers for the product P and the same for the running sum. K advances in stages of 64
// (one pair of sub-blocks = 32 quant bytes of a row): a lane (row n, half h) fetches the 16 quant bytes [16 h, 16 h + 16) of
// the pair (Q8_0: codes of each of the two blocks) straight into registers, expands them into the B operands of the stage's four MFMA k-steps
// (low nibbles: k-steps 0, 1; high nibbles: 2, 3), and the token rows of the stage (64 halves each) are copied global -> LDS
// three stages ahead through a 4-stage ring shared by the workgroup's waves (the 16-byte pieces of a row XOR-swizzled by (row / 2) % 8:
// sixteen consecutive rows then cover all banks, and a copy instruction still writes 1 KB of consecutive LDS).
// One barrier per stage, in its middle, so that the stream of
// operand requests and MFMAs runs on over the stages' borders, and the expansions, the folds of a product and the requests stand
// between the MFMAs (333 rows 194.6 -> 191.7 us, 4096 rows over 256 experts 3.66 -> 3.59 ms).
// MODE 0 pairs gate row f with up row f in lanes n and n + 16 of one wave, so SwiGLU needs one 16-lane exchange.
// What bounds it: with whole tiles of 128 rows a SIMD takes 38 ns a product (one such product after the other on random operands, out of
// registers, takes it 20 ns at the clock that the chip's power leaves, with seven vector instructions beside each 26); with few rows
// the weights' way to the registers. Q5_K and Q8_0 rows, through LDS by loader waves before (layer, top-8): hidden 2048 / ffn 768 / 128
// experts, 100, 333, 1000, 4000 rows Q5_K 255, 353, 535, 1438 -> 134, 206, 341, 914 us, Q8_0 252, 335, 521, 1468 -> 184, 257, 348, 979;
// 4096 rows of hidden 4096 / ffn 2048 / 64 experts 4720 -> 3409, 4994 -> 3830 (Q4_K 2857).
#pragma once
#include "device_math.hpp"
#include "prefill_args.hpp"
#include "q4k_rows.hpp"
#include <type_traits>

namespace strix950 {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) uint8_t pf_lds;

// the status word of an assignment's row, and the first of its `features` unweighted outputs
__device__ __forceinline__ uint32_t* pf_status_of(const PrefillArgs& a, uint32_t assignment) {
    return reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(a.status) + static_cast<size_t>(assignment / a.top_k) * a.status_rs);
}
__device__ __forceinline__ float* pf_rawdots_of(const PrefillArgs& a, uint32_t assignment) {
    if (a.rawdots_rs == 0) return a.rawdots + static_cast<size_t>(assignment) * a.features;
    const uint32_t row = assignment / a.top_k, slot = assignment - row * a.top_k;
    return reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.rawdots) + static_cast<size_t>(row) * a.rawdots_rs) + static_cast<size_t>(slot) * a.features;
}
// include/strix/moe/combine.hpp:24-33 (the stored output of a bfloat16 Linear: nearest even, a NaN as it is)
__device__ __forceinline__ float pf_round_bf16(float x) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, x);
    if ((bits & 0x7f800000U) == 0x7f800000U && (bits & 0x7fffffU)) return x;
    return __builtin_bit_cast(float, (bits + 0x7fffU + ((bits >> 16U) & 1U)) & 0xffff0000U);
}

__device__ __forceinline__ uint32_t pack_half2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2v{a, b}, half2v));      // v_cvt_pk_f16_f32: round to nearest even
}
// v -> fp16 hi = fp16(v), lo = fp16(v - hi)
__device__ __forceinline__ void split_half(float v, _Float16& hi, _Float16& lo) {
    hi = static_cast<_Float16>(v);
    lo = static_cast<_Float16>(v - static_cast<float>(hi));
}

// Workgroup barrier that orders LDS traffic only. __syncthreads() also waits for every outstanding global memory operation
// of the wave, which would drain the copies and fetches that are in flight for later steps at every barrier; their
// arrival is awaited explicitly where it is needed.
// (A fence on the LDS address space counts the copies' LDS writes and waits for them too, hence the plain instructions:
// LDS stores of this wave complete, barrier; the compiler moves no memory access across the statement.)
__device__ __forceinline__ void pf_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Token copies a wave issues per stage: one 1 KB copy per plane (h hi and lo at once: two) and 8 WAVES rows of the live token tiles.
template <uint32_t PLANES, uint32_t WAVES> __host__ __device__ constexpr uint32_t rg_token_ops(uint32_t live) {
    return PLANES * ((32U * live + 8U * WAVES - 1U) / (8U * WAVES));
}
enum { kRgQ4K = 0, kRgQ80 = 1, kRgQ5K = 2 };
// Number of vector-memory operations a wave issues in stage p (= stage % 4) of every super-block: the nt token copies of the
// stage three ahead, one quant fetch (Q8_0: three operations), and the header fetch (p = 0; Q5_K: and the fifth bits) or the sums copy (p = 1).
// whole: the quants of the next super-block all at once with its header (p = 0).
__host__ __device__ constexpr uint32_t rg_stage_ops(int fmt, uint32_t nt, uint32_t p, bool whole) {
    const uint32_t head = fmt == kRgQ5K ? 2U : 1U;
    return fmt == kRgQ80 ? nt + 3U : nt + (p == 0U ? head : p == 1U ? 1U : 0U) + (!whole ? 1U : p == 0U ? 4U : 0U);
}

// One global -> LDS copy of 16 bytes per lane (lane l lands at lds_at + 16 l, lds_at a scalar), issued as plain instructions: the
// compiler is not told about it, so it adds no waits of its own around later LDS reads; the arrival of a copy is awaited
// by a counted s_waitcnt before the barrier that publishes the stage.
__device__ __forceinline__ void copy16_to_lds_at(const uint8_t* src, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_at), "v"(src) : "memory", "m0");
}
// four bytes per lane (lane l lands at lds_at + 4 l)
__device__ __forceinline__ void copy4_to_lds_at(const uint32_t* src, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(lds_at), "v"(src) : "memory", "m0");
}

struct Rg8 { u32x4 a, b; uint32_t e; };                   // Q8_0: a stage's words of a lane
struct RgFactor { half2v mul, add; };

// Waits until at most N younger operations are out, for the registers that follow (FIRST: the first of them as well)
template <uint32_t N, bool FIRST> __device__ __forceinline__ void rg_wait_for(u32x4& f, u32x4& a, u32x4& b) {
    if (FIRST) asm volatile("s_waitcnt vmcnt(%3)" : "+v"(f), "+v"(a), "+v"(b) : "n"(N) : "memory");
    else asm volatile("s_waitcnt vmcnt(%2)" : "+v"(a), "+v"(b) : "n"(N) : "memory");
}
template <uint32_t N, bool FIRST> __device__ __forceinline__ void rg_wait_for(u32x4& f, u32x4& a, u32x4& b, u32x4& c, u32x4& d, u32x4& e) {
    if (FIRST) asm volatile("s_waitcnt vmcnt(%6)" : "+v"(f), "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e) : "n"(N) : "memory");
    else asm volatile("s_waitcnt vmcnt(%5)" : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e) : "n"(N) : "memory");
}
template <int N> __device__ __forceinline__ void rg_wait() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

// WAVES: 8 (one workgroup per compute unit, items of up to 128 rows) or 4 (three workgroups, 32 rows at a time: batches whose experts hold
// few rows are bound by how many weight bytes are asked for at once, and 160 registers let a third workgroup ask).
// WHOLE: the four-wave form asks for a super-block's header and quants in one go, a super-block ahead: the 144 bytes of a row are two
// cache lines, which the wide form's four fetches, a stage apart, bring from the L2 four times (its registers leave no room for the copy;
// 300 rows of hidden 5120 / ffn 1536 / 160 experts 763 -> 700 us).
template <int MODE, uint32_t WAVES, int FMT>
__global__ __launch_bounds__(64 * WAVES, WAVES == 4U ? 3 : 2) void prefill_reg_kernel(PrefillArgs a, uint32_t items_at, uint32_t order_at) {
    constexpr uint32_t TOKENS = WAVES == 4U ? 32U : 128U;
    static_assert(TOKENS <= 16U * WAVES && TOKENS % (8U * WAVES) == 0, "one sums copy per wave, a token copy of 8 rows per wave and part");
    constexpr bool WHOLE = WAVES == 4U && FMT != kRgQ80;
    // SCALED: the operand of a Q4_K weight is 2^-14 sc q, as the packed product of a subnormal (the nibble where it lies in its byte: 2^-24 q or 2^-20 q)
    // and 2^10 sc or 2^6 sc: exact, no shift for the high nibbles, and no 1024 to take out of the sum again.
    constexpr bool SCALED = FMT == kRgQ4K;
    // Q8_0: stages of weights in registers. The wide form has room for two beside its sums (14 registers of the gate / up rows and 9 of the
    // down rows are spilled at a unit's start and read at its end, as 7 and 5 of Q4_K and Q5_K are; with four stages 110, inside the K loop: 1000 rows of hidden
    // 2048 / ffn 768 / 128 experts 342 -> 435 us).
    constexpr uint32_t RING8 = WAVES == 4U ? 4U : 2U;
    constexpr uint32_t BLOCK = FMT == kRgQ5K ? 176U : 144U, QUANTS_AT = FMT == kRgQ5K ? 48U : 16U;          // of a K-quant super-block
    // h enters as fp16 hi + lo. Q4_K: both planes in one sweep of the weights, two products per operand. Q5_K and Q8_0: K is swept twice, lo
    // first: the hi products then round as they would alone (these formats follow the exact product to 1e-7, where a rounding more per
    // product shows: rms error of Q5_K rows 0.99e-7, 1.17e-7 with both planes in one sum).
    constexpr uint32_t SWEEPS = MODE == 1 && FMT != kRgQ4K ? 2U : 1U;
    constexpr uint32_t PLANES = MODE == 1 && SWEEPS == 1U ? 2U : 1U, TILES = TOKENS / 32U, PART_ROWS = 8U * WAVES;
    constexpr uint32_t STAGE = TOKENS * 128U;                     // one plane of one stage: TOKENS rows x 64 halves
    __shared__ __attribute__((aligned(16))) uint8_t tok0[PLANES * STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t tok1[PLANES * STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t tok2[PLANES * STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t tok3[PLANES * STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t s_tile_mem[2][TOKENS * 64U];           // [token][hi 16 | lo 16] sums of 16 sub-blocks
    __shared__ float part_sum[WAVES][TOKENS];                                              // MODE 0 epilogue: a wave's 16-feature sums of h
    pf_lds* const tok_stage[4] = {(pf_lds*)tok0, (pf_lds*)tok1, (pf_lds*)tok2, (pf_lds*)tok3};
    pf_lds* const s_tile = (pf_lds*)s_tile_mem;

    // LIST: the workgroup's units, up to 64 at a time, are listed in LDS (expert, first row in plan order, rows, feature tile), and the assignments of a
    // unit's rows are there before it starts. Asked for one after the other in front of a unit's first copy, item and assignments are two trips to
    // memory that nothing hides, and the stores at its end wait for a third: 1000 rows of hidden 2048 / ffn 768 / 128 experts 291 -> 268 us, 4096 rows
    // of hidden 4096 / ffn 2048 / 256 experts 3932 -> 3806. The four-wave form has one to three units a workgroup and two more of them beside
    // it: the list costs it more than it saves (64 rows 95.9 -> 97.9 us), and so did copies that run on from a unit into the next (97.4; 333
    // rows 162.2 -> 158.8, Q8_0 rows 169.5 -> 173.6).
    constexpr bool LIST = WAVES == 8U;
    __shared__ __attribute__((aligned(16))) uint4 unit_mem[LIST ? 64U : 1U];
    __shared__ uint32_t unit_count;
    __shared__ uint32_t order_mem[2][LIST ? TOKENS : 1U];
    static_assert(!LIST || TOKENS % 64U == 0, "copies of whole waves");

    if (MODE == 1 && (*a.job_status & MI355_STATUS_NONFINITE_PROJECTION)) return;
    const uint32_t* order = a.plan + order_at;
    const uint32_t lane = threadIdx.x & 63U, wave = threadIdx.x >> 6, n31 = lane & 31U, half = lane >> 5;
    const uint32_t wave_s = __builtin_amdgcn_readfirstlane(wave);       // the wave's number as a scalar (LDS addresses of its copies)
    const uint32_t blocks = a.k / 256U, last_block = SWEEPS * blocks - 1U, stages = a.k / 64U, last_stage = SWEEPS * stages - 1U;
    const uint32_t last_group = (blocks + 1U) / 2U - 1U;
    const size_t to_hi = SWEEPS == 2U ? reinterpret_cast<uintptr_t>(a.h) - reinterpret_cast<uintptr_t>(a.h_lo) : 0U;      // (modulo 2^64)
    const size_t sum_row = pf_sum_row_bytes(a.k);

    // Wide: the tiles of an item run on one XCD, whose L2 then holds its token rows. Four waves: few rows per item, whose units differ in
    // length more than their token rows cost: an item's tiles go round the XCDs (of the items that were made). An item holds at most
    // TOKENS rows in either form (prefill_split).
    constexpr bool ROUND = WAVES == 4U;
    const uint32_t units = ROUND ? a.plan[4] * a.tiles : a.units;
    const auto item_of = [&](uint32_t unit) {           // (a unit that does not exist: no rows)
        const uint32_t q = unit >> 3;
        const uint32_t item_index = ROUND ? unit / a.tiles : (q / a.tiles) * 8U + (unit & 7U), at = (ROUND ? unit : q) % a.tiles;
        uint4 item = {0U, 0U, 0U, 0U};
        if (unit < units && item_index < a.items) item = *reinterpret_cast<const uint4*>(a.plan + items_at + 4U * item_index);
        return uint4{item.x, item.y, item.y < item.z ? item.z - item.y : 0U, at};
    };
    const auto copy_assignments = [&](uint32_t u) {     // of listed unit u (past its rows: the last one's again)
        if (wave_s >= TOKENS / 64U) return;
        const uint4 item = unit_mem[u];
        copy4_to_lds_at(order + item.y + (threadIdx.x < item.z ? threadIdx.x : item.z - 1U),
                        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((pf_lds*)order_mem[u & 1U])) + 256U * wave_s);
    };
    for (uint32_t base = blockIdx.x; base < units; base += (LIST ? 64U : 1U) * gridDim.x) {
    uint32_t listed = 1;
    if constexpr (LIST) {
        if (threadIdx.x < 64U) {
            const uint4 item = item_of(base + lane * gridDim.x);
            const uint64_t lives = __ballot(item.z != 0U);
            if (item.z) unit_mem[__popcll(lives & ((1ULL << lane) - 1ULL))] = item;
            if (lane == 0U) unit_count = __popcll(lives);
        }
        pf_barrier();
        listed = __builtin_amdgcn_readfirstlane(unit_count);
        if (listed) copy_assignments(0);
        rg_wait<0>();
        pf_barrier();                                   // (and unit_count is free again)
    }
    for (uint32_t u = 0; u < listed; ++u) {
    const uint4 item = LIST ? unit_mem[u] : item_of(base);
    const uint32_t e = __builtin_amdgcn_readfirstlane(item.x), begin = __builtin_amdgcn_readfirstlane(item.y);
    const uint32_t count = __builtin_amdgcn_readfirstlane(item.z), tile = __builtin_amdgcn_readfirstlane(item.w);
    if (!LIST && count == 0U) continue;
    const uint32_t* const assignment = LIST ? order_mem[u & 1U] : order + begin;
    if (LIST && u + 1U < listed) copy_assignments(u + 1U);              // (older than every counted copy; awaited at the unit's end)

    // ---- the lane's weight row
    uint32_t feature;                                  // MODE 0: gate (n31 < 16) / up feature; MODE 1: output column
    const uint8_t* wbase = a.wa;
    if (MODE == 0) { feature = tile * (16U * WAVES) + 16U * wave + (n31 & 15U); if (n31 & 16U) wbase = a.wb; }
    else feature = tile * (32U * WAVES) + 32U * wave + n31;
    const uint8_t* wrow = wbase + static_cast<size_t>(e) * a.expert_stride + static_cast<size_t>(feature) * a.row_stride;

    // ---- token copies: part i of a stage moves tile rows PART_ROWS i + 8 wave .. + 8 (of both planes: MODE 1); lane = (row % 8, slot)
    constexpr uint32_t PARTS = TOKENS / PART_ROWS;
    const uint8_t* tsrc[PLANES][PARTS];
#pragma unroll
    for (uint32_t i = 0; i < PARTS; ++i) {
        const uint32_t row = PART_ROWS * i + 8U * wave + (lane >> 3), tok = row < count ? row : count - 1U;
        const uint32_t piece = (lane & 7U) ^ ((row >> 1) & 7U);
        if (MODE == 0) tsrc[0][i] = a.x + static_cast<size_t>(assignment[tok] / a.top_k) * a.x_stride + 16U * piece;
        else {
            // (h rows past the item's are other items' rows or the padding rows of the workspace: read, multiplied and never stored)
            const size_t from = static_cast<size_t>(begin + row) * a.k;
            if (PLANES == 2U) tsrc[0][i] = reinterpret_cast<const uint8_t*>(a.h + from) + 16U * piece;
            tsrc[PLANES - 1U][i] = reinterpret_cast<const uint8_t*>(a.h_lo + from) + 16U * piece;
        }
    }
    // ---- sums copy: piece = (token, part): parts 0, 1 = hi halves 0-7 / 8-15, parts 2, 3 = lo
    const uint8_t* ssrc;
    {
        const uint32_t row = (threadIdx.x >> 2) & (TOKENS - 1U), part = threadIdx.x & 3U, tok = row < count ? row : count - 1U;
        const uint8_t* base = MODE == 0 ? a.x_sums + static_cast<size_t>(assignment[tok] / a.top_k) * sum_row
                                        : a.h_sums + static_cast<size_t>(begin + tok) * sum_row;
        ssrc = base + 16U * (part & 1U) + (part >> 1) * (sum_row / 2U);
    }
    const auto copy_sums = [&](uint32_t g) {
        const uint32_t gc = g < last_group ? g : last_group;
        copy16_to_lds_at(ssrc + static_cast<size_t>(gc) * 32U,
                         static_cast<uint32_t>(reinterpret_cast<uintptr_t>(s_tile)) + (g & 1U) * (TOKENS * 64U) + 1024U * (wave_s & (TOKENS / 16U - 1U)));
    };
    // block / stage of the rows that block b / stage s of the sweeps is (past the end: the last)
    const auto block_of = [&](uint32_t b) { const uint32_t c = b < last_block ? b : last_block; return SWEEPS == 2U && c >= blocks ? c - blocks : c; };
    const auto stage_of = [&](uint32_t s) { const uint32_t c = s < last_stage ? s : last_stage; return SWEEPS == 2U && c >= stages ? c - stages : c; };
    const auto fetch_header = [&](uint32_t b, u32x4& hd, u32x4& fifth) {
        const uint8_t* blk = wrow + static_cast<size_t>(block_of(b)) * BLOCK;
        asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(hd) : "v"(blk) : "memory");
        if (FMT == kRgQ5K) {                           // of elements 16 half .. + 16 of every sub-block
            const uint8_t* bits = blk + 16U + 16U * half;
            asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(fifth) : "v"(bits) : "memory");
        }
    };
    // the quants of stage 4 b + p (an offset from the super-block's one address, which costs less than an address a stage)
    const auto fetch_quants = [&](uint32_t b, auto p, u32x4& qs) {
        const uint8_t* at = wrow + static_cast<size_t>(block_of(b)) * BLOCK + 16U * half;
        asm volatile("global_load_dwordx4 %0, %1, off offset:%2" : "=v"(qs) : "v"(at), "n"(QUANTS_AT + 32U * decltype(p)::value) : "memory");
    };
    const auto fetch_whole = [&](uint32_t b, u32x4 (&q)[4]) {           // of a super-block
        fetch_quants(b, std::integral_constant<uint32_t, 0>{}, q[0]);
        fetch_quants(b, std::integral_constant<uint32_t, 1>{}, q[1]);
        fetch_quants(b, std::integral_constant<uint32_t, 2>{}, q[2]);
        fetch_quants(b, std::integral_constant<uint32_t, 3>{}, q[3]);
    };

    // Q8_0: a stage is two blocks (fp16 d, 32 codes; 34 bytes), 68 bytes from a 4-byte boundary. The lane's 16 codes of the first lie two
    // bytes past a word (four words and the next), those of the second on one. Its words hold d of the first block (half 0: in front of the
    // codes) or of the second (half 1: behind them).
    const auto fetch_blocks = [&](uint32_t s, Rg8& r) {
        const uint8_t* first = wrow + 68U * stage_of(s) + 16U * half;
        // (the registers are named as read, so that they stay the same ones from fetch to fetch)
        asm volatile("global_load_dwordx4 %0, %1, off" : "+v"(r.a) : "v"(first) : "memory");
        asm volatile("global_load_dword %0, %1, off offset:16" : "+v"(r.e) : "v"(first) : "memory");
        asm volatile("global_load_dwordx4 %0, %1, off offset:36" : "+v"(r.b) : "v"(first) : "memory");
    };

    // ---- expansion: 8 nibbles (low or high) of two quant words -> the B operand of one k-step: four registers of two fp16
    // numbers each
    uint32_t magic;
    asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
    // Q5_K: sc q is up to 1953, past the offset's mantissa: fma(1024 + q, sc, -1024 sc) = sc q, exact. Q8_0: 1152 + code, minus 1152.
    const _Float16 minus = static_cast<_Float16>(-1152.0F);
    // two weights: bytes 0, 1 or (odd) 2, 3 of a word
    const auto expand_pair = [&](uint32_t w, uint32_t odd, const RgFactor& f) -> uint32_t {
        if (SCALED) return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0U, w, odd ? 0x0c030c02U : 0x0c010c00U)) * f.mul);
        const half2v t = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(magic, w, odd ? 0x05030502U : 0x05010500U));
        if (FMT == kRgQ5K) return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t, f.mul, f.add));
        return __builtin_bit_cast(uint32_t, t + half2v{minus, minus});
    };
    const auto expand = [&](uint32_t w0, uint32_t w1, const RgFactor& f) -> half8 {
        return __builtin_bit_cast(half8, u32x4{expand_pair(w0, 0U, f), expand_pair(w0, 1U, f), expand_pair(w1, 0U, f), expand_pair(w1, 1U, f)});
    };
    // a word of four nibbles (Q5_K: with their fifth bits, bit `bit` of each byte of f)
    const auto low = [&](uint32_t w, uint32_t f, uint32_t bit) -> uint32_t {
        return (w & 0x0f0f0f0fU) | (FMT == kRgQ5K ? ((f >> bit) & 0x01010101U) << 4 : 0U);
    };
    const auto high = [&](uint32_t w, uint32_t f, uint32_t bit) -> uint32_t { return SCALED ? w & 0xf0f0f0f0U : low(w >> 4, f, bit); };
    // four bytes of the packed six-bit factors as fp16 integers, bytes 0 and 1 or (odd) 2 and 3 in a register
    const auto six_bits = [&](uint32_t m, uint32_t odd) -> half2v {
        const half2v offset = {static_cast<_Float16>(-1024.0F), static_cast<_Float16>(-1024.0F)};
        return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(magic, m, odd ? 0x05030502U : 0x05010500U)) + offset;
    };
    // SCALED: 2^10 sc of sub-block 2 p and 2^6 sc of 2 p + 1
    half2v scaled[4];
    const auto set_scaled = [&](const u32x4& hd) {
        const uint32_t first = hd.y & 0x3f3f3f3fU, last = (hd.w & 0x0f0f0f0fU) | ((hd.y >> 2) & 0x30303030U);
        const half2v units = {static_cast<_Float16>(1024.0F), static_cast<_Float16>(64.0F)};
#pragma unroll
        for (uint32_t q = 0; q < 4U; ++q) scaled[q] = six_bits(q < 2U ? first : last, q & 1U) * units;
    };
    // of sub-block 2 p or (odd) 2 p + 1; SCALED: of the header that set_scaled was given (Q5_K: src/cpu/core/routed_expert.cpp:65-71)
    const auto factor_of = [&](const u32x4& hd, uint32_t p, uint32_t odd) -> RgFactor {
        RgFactor f{};
        if (SCALED) f.mul = odd ? half2v{scaled[p].y, scaled[p].y} : half2v{scaled[p].x, scaled[p].x};
        else if (FMT == kRgQ5K) {
            const uint32_t at = 16U * (p & 1U) + 8U * odd, first = (hd.y >> at) & 255U, last = (hd.w >> at) & 255U;
            const uint32_t sc = p < 2U ? (first & 63U) : ((last & 15U) | ((first >> 6) << 4));
            const _Float16 c = static_cast<_Float16>(static_cast<float>(sc)), n = c * static_cast<_Float16>(-1024.0F);
            f.mul = half2v{c, c};
            f.add = half2v{n, n};
        }
        return f;
    };
    // Q8_0: words 2 k, 2 k + 1 of the lane's codes of the stage's first block, as unsigned bytes code + 128
    const auto first_codes = [&](const Rg8& r, uint32_t k, uint32_t& w0, uint32_t& w1) {
        w0 = __builtin_amdgcn_alignbyte(k ? r.a.w : r.a.y, k ? r.a.z : r.a.x, 2U) ^ 0x80808080U;
        w1 = __builtin_amdgcn_alignbyte(k ? r.e : r.a.z, k ? r.a.w : r.a.y, 2U) ^ 0x80808080U;
    };

    // Everything from the first fetch to the last store is instantiated per number of token tiles that hold a row of the item
    // (the other tiles are neither read nor multiplied). The weight fetches are plain instructions the compiler does not
    // track, so a register they write must stay reserved until the fetch has landed - including the (clamped) fetches of a
    // unit's last stages that nothing uses: they are awaited at the end of the instantiation, and no fetched register is
    // live across a join of two instantiations (a join may copy registers, and a copy of a register whose fetch is still in
    // flight would copy stale data).
    const auto run_unit = [&](auto live_constant) __attribute__((always_inline)) {
    constexpr uint32_t LIVE = decltype(live_constant)::value, NT = rg_token_ops<PLANES, WAVES>(LIVE);
    const auto copy_tokens = [&](uint32_t s, pf_lds* stage) {
        const uint32_t sc = stage_of(s);
        const size_t plane = SWEEPS == 2U && s >= stages ? to_hi : 0U;
        const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(stage)) + 1024U * wave_s;
#pragma unroll
        for (uint32_t i = 0; i < NT; ++i)
            copy16_to_lds_at(tsrc[i % PLANES][i / PLANES] + (plane + static_cast<size_t>(sc) * 128U), base + (i % PLANES) * STAGE + 128U * PART_ROWS * (i / PLANES));
    };
    floatx16 acc[LIVE], part[LIVE];
#pragma unroll
    for (uint32_t i = 0; i < LIVE; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) { acc[i][j] = 0.0F; part[i][j] = 0.0F; }
    const uint32_t trow = n31 * 128U, sw = (n31 >> 1) & 7U;
    uint32_t piece_at[4];                              // k-step j reads piece (j >= 2 ? 4 : 0) + 2 half + (j & 1) of the lane's token row
#pragma unroll
    for (uint32_t j = 0; j < 4U; ++j) piece_at[j] = ((((j >> 1) << 2) + 2U * half + (j & 1U)) ^ sw) << 4;

    // ---- prologue: the operations of "stages -3, -2, -1" in the loop's own order, so that its counts hold from the first
    // stage on; before them the header and the quants of stage 0
    u32x4 hd_cur, hd_next = {0U, 0U, 0U, 0U}, f_cur = {0U, 0U, 0U, 0U}, f_next = {0U, 0U, 0U, 0U}, qs[4], qn[4];   // (qn: the next super-block's quants, WHOLE only)
    Rg8 q8[RING8];
    if (FMT == kRgQ80) {
#pragma unroll
        for (uint32_t r = 0; r < RING8; ++r) q8[r] = Rg8{{0U, 0U, 0U, 0U}, {0U, 0U, 0U, 0U}, 0U};
    }
    float d_last = 0.0F;                                               // Q8_0: d of the last block of the stage before
    if constexpr (FMT == kRgQ80) {
        fetch_blocks(0, q8[0]);
        copy_tokens(0, tok_stage[0]);
        if (RING8 == 4U) fetch_blocks(1, q8[1]);
        copy_tokens(1, tok_stage[1]);
        if (RING8 == 4U) fetch_blocks(2, q8[2 % RING8]);
        copy_tokens(2, tok_stage[2]);
        fetch_blocks(RING8 - 1U, q8[RING8 - 1U]);
        // younger than the token copies of stage 0: three fetches and two stages of NT. A ring of two fetches less in the first stages than
        // the loop counts on: the copies of stage 1 are awaited here as well
        asm volatile("s_waitcnt vmcnt(%3)" : "+v"(q8[0].a), "+v"(q8[0].b), "+v"(q8[0].e) : "n"(RING8 == 4U ? 2U * NT + 9U : NT + 3U) : "memory");
    } else if constexpr (WHOLE) {
        fetch_header(0, hd_cur, f_cur);
        fetch_whole(0, qs);
        copy_tokens(0, tok_stage[0]); copy_sums(0);
        copy_tokens(1, tok_stage[1]);
        copy_tokens(2, tok_stage[2]);
        // younger than the token copies and sums of stage 0: two stages of NT
        rg_wait_for<2U * NT, FMT == kRgQ5K>(f_cur, hd_cur, qs[0], qs[1], qs[2], qs[3]);
    } else {
        fetch_header(0, hd_cur, f_cur); fetch_quants(0, std::integral_constant<uint32_t, 0>{}, qs[0]);
        copy_tokens(0, tok_stage[0]); copy_sums(0); fetch_quants(0, std::integral_constant<uint32_t, 1>{}, qs[1]);
        copy_tokens(1, tok_stage[1]); fetch_quants(0, std::integral_constant<uint32_t, 2>{}, qs[2]);
        copy_tokens(2, tok_stage[2]); fetch_quants(0, std::integral_constant<uint32_t, 3>{}, qs[3]);
        // younger than the token copies of stage 0: sums + quants, then two stages of NT + 1
        rg_wait_for<2U * NT + 4U, FMT == kRgQ5K>(f_cur, hd_cur, qs[0]);
    }
    pf_barrier();

    half8 bfrag;                                       // B operand of the next k-step
    if constexpr (FMT == kRgQ80) {
        uint32_t w0, w1;
        first_codes(q8[0], 0U, w0, w1);
        bfrag = expand(w0, w1, RgFactor{});
    } else {
        if (SCALED) set_scaled(hd_cur);
        bfrag = expand(low(qs[0].x, f_cur.x, 0U), low(qs[0].y, f_cur.y, 0U), factor_of(hd_cur, 0U, 0U));
    }
    // A stage's MFMAs as a flat sequence of slots m = (k-step j, plane, token tile i); the A operand of slot m + W is requested right after
    // the MFMA of slot m into the registers that MFMA has just read (a window of W operands, which runs on over the stages' borders).
    constexpr uint32_t PER = PLANES * LIVE, N = 4U * PER, W = N / 2U < 4U ? N / 2U : 4U;
    half8 frag[W];
    const auto request = [&](uint32_t m, const pf_lds* stage) __attribute__((always_inline)) {
        const uint32_t j = m / PER, pl = (m / LIVE) % PLANES, i = m % LIVE;
        frag[m % W] = *reinterpret_cast<const __attribute__((address_space(3))) half8*>(stage + trow + pl * STAGE + i * 32U * 128U + piece_at[j]);
    };
#pragma unroll
    for (uint32_t m = 0; m < W; ++m) request(m, tok_stage[0]);

    {
        const auto stage = [&](auto p_constant, uint32_t b) __attribute__((always_inline)) {
                constexpr uint32_t p = decltype(p_constant)::value;
                const uint32_t s = 4U * b + p, bb = SWEEPS == 2U && b >= blocks ? b - blocks : b;            // (bb: of the rows)
                const RgFactor f_lo = factor_of(hd_cur, p, 0U), f_hi = factor_of(hd_cur, p, 1U);
                const u32x4 qw = qs[p];
                const Rg8 r8 = q8[p % RING8];
                const float d_now = half_bits_to_float(hd_cur.x & 0xffffU) * (SCALED ? 16384.0F : 1.0F);
                float d_first = 0.0F, d_second = 0.0F;                                   // Q8_0: of the stage's two blocks
                if (FMT == kRgQ80) {
                    const uint32_t mine = half ? r8.e >> 16 : r8.a.x & 0xffffU;
                    const auto both = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);
                    d_first = half_bits_to_float(both[0]);
                    d_second = half_bits_to_float(both[1]);
                }
                const auto fold = [&](uint32_t i, float d) __attribute__((always_inline)) {   // end of a super-block (Q8_0: block): running sum += d * P
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][r] = __builtin_fmaf(d, part[i][r], acc[i][r]);
                };
                half8 bcur = bfrag;
                u32x4 bnext = __builtin_bit_cast(u32x4, bfrag);
                uint32_t nw0 = 0, nw1 = 0;                     // the next k-step's quant words and factor
                RgFactor nf{};
#pragma unroll
                for (uint32_t m = 0; m < N; ++m) {
                    const uint32_t j = m / PER, i = m % LIVE;
                    if (m % PER == 0) {
                        // a new k-step: take its B operand; the next one's is expanded between this one's MFMAs
                        bcur = __builtin_bit_cast(half8, bnext);
                        if (j == 0) {
                            if (FMT == kRgQ80) first_codes(r8, 1U, nw0, nw1);
                            else { nw0 = low(qw.z, f_cur.z, 2U * p); nw1 = low(qw.w, f_cur.w, 2U * p); nf = f_lo; }
                        } else if (j == 1) {
                            if (FMT == kRgQ80) { nw0 = r8.b.x ^ 0x80808080U; nw1 = r8.b.y ^ 0x80808080U; }
                            else { nw0 = high(qw.x, f_cur.x, 2U * p + 1U); nw1 = high(qw.y, f_cur.y, 2U * p + 1U); nf = f_hi; }
                        } else if (j == 2) {
                            if (FMT == kRgQ80) { nw0 = r8.b.z ^ 0x80808080U; nw1 = r8.b.w ^ 0x80808080U; }
                            else { nw0 = high(qw.z, f_cur.z, 2U * p + 1U); nw1 = high(qw.w, f_cur.w, 2U * p + 1U); nf = f_hi; }
                            // The stage's middle: its token copies' turn. The tokens of stage s + 1 were copied two stages ago (younger: the rest
                            // of that stage's operations and the next one's); behind the barrier every wave's have landed, and every wave
                            // has read the last of stage s - 1, whose slot takes stage s + 3. (At a stage's border the barrier made both waves
                            // of a SIMD wait for their first operands at once.)
                            rg_wait<static_cast<int>(rg_stage_ops(FMT, NT, (p + 2U) & 3U, WHOLE) - NT + rg_stage_ops(FMT, NT, (p + 3U) & 3U, WHOLE))>();
                            asm volatile("s_barrier" ::: "memory");
                            copy_tokens(s + 3U, tok_stage[(p + 3U) & 3U]);
                            if (FMT == kRgQ80) {
                                asm volatile("" : "+v"(nw0), "+v"(nw1));         // (worked out before their registers are fetched anew)
                                fetch_blocks(s + RING8, q8[p % RING8]);
                            }      // the stage's quant registers are free now
                            else {
                                if (p == 1) copy_sums(SWEEPS == 2U && b + 1U == blocks ? 0U : (bb >> 1) + 1U);
                                if (!WHOLE) fetch_quants(b + 1U, p_constant, qs[p]);
                                if (p == 0) fetch_header(b + 1U, hd_next, f_next);
                            }
                            if (WHOLE && p == 0) fetch_whole(b + 1U, qn);
                        } else {
                            // first k-step of the next stage: its quants (the next super-block's header with them) were fetched in stage s - 3
                            // (WHOLE: all of the next super-block's in stage 0); younger the three stages since
                            constexpr uint32_t pn = (p + 1U) & 3U;
                            constexpr uint32_t younger = rg_stage_ops(FMT, NT, (p + 2U) & 3U, WHOLE) + rg_stage_ops(FMT, NT, (p + 3U) & 3U, WHOLE) + rg_stage_ops(FMT, NT, p, WHOLE);
                            if constexpr (FMT == kRgQ80) {
                                Rg8& next8 = q8[pn % RING8];
                                asm volatile("s_waitcnt vmcnt(%3)" : "+v"(next8.a), "+v"(next8.b), "+v"(next8.e) : "n"((RING8 - 1U) * (NT + 3U)) : "memory");
                                first_codes(next8, 0U, nw0, nw1);
                            } else {
                                if (WHOLE) {
                                    if (p == 3U) {
                                        rg_wait_for<younger, FMT == kRgQ5K>(f_next, hd_next, qn[0], qn[1], qn[2], qn[3]);
#pragma unroll
                                        for (uint32_t q4 = 0; q4 < 4U; ++q4) qs[q4] = qn[q4];
                                    }
                                } else if (p == 3U) rg_wait_for<younger, FMT == kRgQ5K>(f_next, hd_next, qs[pn]);
                                else asm volatile("s_waitcnt vmcnt(%1)" : "+v"(qs[pn]) : "n"(younger) : "memory");
                                if (SCALED && p == 3U) set_scaled(hd_next);
                                const u32x4 fb = p == 3U ? f_next : f_cur;
                                nw0 = low(qs[pn].x, fb.x, 2U * pn); nw1 = low(qs[pn].y, fb.y, 2U * pn); nf = factor_of(p == 3U ? hd_next : hd_cur, pn, 0U);
                            }
                        }
                    }
                    if (FMT == kRgQ80 ? m % (2U * PER) < LIVE : p == 0 && m < LIVE) {     // first MFMA of a super-block's (Q8_0: block's) product: it starts from zero
                        const floatx16 zero = {0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F, 0.0F};
                        part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[m % W], bcur, zero, 0, 0, 0);
                    } else {
                        part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag[m % W], bcur, part[i], 0, 0, 0);
                    }
                    if (m + W < N) request(m + W, tok_stage[p]);
                    else request(m + W - N, tok_stage[(p + 1U) & 3U]);
                    // this slot's share of the next k-step's four operand registers
#pragma unroll
                    for (uint32_t q = 4U * (m % PER) / PER; q < 4U * (m % PER + 1U) / PER; ++q)
                        bnext[q] = expand_pair(q < 2U ? nw0 : nw1, q & 1U, nf);
                    if (FMT == kRgQ80) {                             // the tile whose next block's product the next slot starts
                        const uint32_t next = (m + 1U) % N;
                        if (next % (2U * PER) < LIVE) fold(next % LIVE, next == 0U ? d_second : next < LIVE ? d_last : d_first);
                    } else if (p == 3U && m > N - LIVE) fold(i - 1U, d_now);       // (the tile before this one's last product is through)
                    // the scheduler otherwise sinks the request down to its use (registers are scarce) and the MFMA then waits
                    // for the whole LDS round trip: nothing moves across this point (1874 -> 1828 us gate / up, 1642 -> 1565 us down)
                    __builtin_amdgcn_sched_barrier(0);
                }
                bfrag = __builtin_bit_cast(half8, bnext);
                d_last = d_second;
                if (FMT != kRgQ80 && p == 3U) {
                    // the super-block's minimums: S hi and S lo (K = 8 + 8; the sums are of hi + lo, once) against the integers m_j, times -dmin
                    const bool least = SWEEPS == 1U || b >= blocks;
                    const pf_lds* st = s_tile + ((bb >> 1) & 1U) * (TOKENS * 64U) + n31 * 64U + 32U * half + 16U * (bb & 1U);
                    const float minus_dmin = -half_bits_to_float(hd_cur.x >> 16);
                    u32x4 mins = {0U, 0U, 0U, 0U};
                    if (least) {
                        const uint32_t first = hd_cur.z & 0x3f3f3f3fU, last = ((hd_cur.w >> 4) & 0x0f0f0f0fU) | ((hd_cur.z >> 2) & 0x30303030U);
#pragma unroll
                        for (uint32_t q = 0; q < 4U; ++q) mins[q] = __builtin_bit_cast(uint32_t, six_bits(q < 2U ? first : last, q & 1U));
                    }
                    const auto minimums = [&](uint32_t i) __attribute__((always_inline)) {
                        const floatx16 zero = {0.0F};
                        return __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const __attribute__((address_space(3))) half8*>(st + i * 32U * 64U), __builtin_bit_cast(half8, mins), zero, 0, 0, 0);
                    };
                    const auto take = [&](uint32_t i, const floatx16& product) __attribute__((always_inline)) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[i][r] = __builtin_fmaf(minus_dmin, product[r], acc[i][r]);
                    };
                    if constexpr (LIVE == 1U) {                      // (registers for both products)
                        if (least) {
                            const floatx16 product = minimums(0);
                            fold(0, d_now);
                            take(0, product);
                        } else fold(0, d_now);
                    } else {
                        fold(LIVE - 1U, d_now);
                        if (least) {
#pragma unroll
                            for (uint32_t i = 0; i < LIVE; ++i) part[i] = minimums(i);
#pragma unroll
                            for (uint32_t i = 0; i < LIVE; ++i) take(i, part[i]);
                        }
                    }
                    hd_cur = hd_next;
                    f_cur = f_next;
                }
        };
        for (uint32_t b = 0; b < SWEEPS * blocks; ++b) {
            stage(std::integral_constant<uint32_t, 0>{}, b);
            stage(std::integral_constant<uint32_t, 1>{}, b);
            stage(std::integral_constant<uint32_t, 2>{}, b);
            stage(std::integral_constant<uint32_t, 3>{}, b);
        }
        if constexpr (FMT == kRgQ80) {                   // the last block's product (of tile 0 folded in the last slot)
#pragma unroll
            for (uint32_t i = 1; i < LIVE; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][r] = __builtin_fmaf(d_last, part[i][r], acc[i][r]);
        }
    }

    // ---- epilogue. Result layout of a 32 x 32 tile: the lane holds weight row n31; register r is token 8 (r / 4) + 4 half + r % 4
    if (MODE == 0) {
        // Lane n31 < 16 holds gate row f of 16 tokens per tile, lane n31 + 16 the up row of the same feature. The two lanes
        // swap halves (the gate lane sends its tokens 8-15, the up lane its tokens 0-7), so each evaluates SwiGLU for eight
        // tokens. This class follows the exact product to a tolerance, so exp and the division are the hardware's
        // (v_exp_f32, v_rcp_f32: one ulp each).
        const uint32_t f_out = tile * (16U * WAVES) + 16U * wave + (n31 & 15U);
        const bool gate_lane = n31 < 16U;
#pragma unroll
        for (uint32_t i = 0; i < LIVE; ++i)
#pragma unroll
            for (uint32_t k = 0; k < 8U; ++k) {
                // (the two registers are named before the per-lane choice: choosing the INDEX per lane instead would make the
                // compiler walk all sixteen registers of the tile with compare-and-select pairs)
                float first = acc[i][k], second = acc[i][8U + k];
                asm volatile("" : "+v"(first), "+v"(second));
                const float sent = gate_lane ? second : first, got = xor16_f(sent);
                const float g = gate_lane ? first : got, u = gate_lane ? got : second;
                const uint32_t r = gate_lane ? k : 8U + k;
                const uint32_t t = 32U * i + 8U * (r / 4U) + 4U * half + (r & 3U);
                const bool live = t < count;
                float gc = g, uc = u;
                swiglu_clamp(gc, uc, a.swiglu_limit);
                const float hv = (gc * __builtin_amdgcn_rcpf(1.0F + __builtin_amdgcn_exp2f(gc * -1.44269504F))) * uc;
                const _Float16 h_hi = static_cast<_Float16>(hv);
                const _Float16 h_lo = static_cast<_Float16>(hv - static_cast<float>(h_hi));
                float sum = live ? static_cast<float>(h_hi) + static_cast<float>(h_lo) : 0.0F;
                sum += xor1_f(sum); sum += xor2_f(sum); sum += xor4_f(sum); sum += xor8_f(sum);     // over the wave's 16 features
                if ((n31 & 15U) == 0) part_sum[wave][t] = sum;    // a sub-block of 32 features is two waves' halves
                if (live) {
                    const size_t at = static_cast<size_t>(begin + t) * a.features + f_out;
                    a.h[at] = h_hi;
                    a.h_lo[at] = h_lo;
                    if (!(finite_f(g) && finite_f(u) && finite_f(static_cast<float>(h_hi)))) {     // h beyond fp16 counts as non-finite
                        atomicOr(pf_status_of(a, assignment[t]), static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
                        atomicOr(a.job_status, static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
                    }
                }
            }
        __syncthreads();
        if (threadIdx.x < WAVES / 2U * TOKENS) {
            const uint32_t t = threadIdx.x & (TOKENS - 1U), pair = threadIdx.x / TOKENS;            // sub-block tile * WAVES / 2 + pair
            if (t < count) {
                const float sum = part_sum[2U * pair][t] + part_sum[2U * pair + 1U][t];
                _Float16* sums = reinterpret_cast<_Float16*>(a.h_sums + static_cast<size_t>(begin + t) * pf_sum_row_bytes(a.features));
                split_half(sum, sums[tile * (WAVES / 2U) + pair], sums[pf_sum_slots(a.features) + tile * (WAVES / 2U) + pair]);
            }
        }
        __syncthreads();                                  // part_sum is free for the next unit
    } else {
        const uint32_t f_out = tile * (32U * WAVES) + 32U * wave + n31;
#pragma unroll
        for (uint32_t i = 0; i < LIVE; ++i)
#pragma unroll
            for (uint32_t r = 0; r < 16U; ++r) {
                const uint32_t t = 32U * i + 8U * (r / 4U) + 4U * half + (r & 3U);
                if (t < count) pf_rawdots_of(a, assignment[t])[f_out] = a.rawdots_bf16 ? pf_round_bf16(acc[i][r]) : acc[i][r];
            }
    }
    if constexpr (FMT == kRgQ80) {
#pragma unroll
        for (uint32_t r = 0; r < RING8; ++r) asm volatile("s_waitcnt vmcnt(0)" : "+v"(q8[r].a), "+v"(q8[r].b), "+v"(q8[r].e) : : "memory");
    } else {
        rg_wait_for<0U, FMT == kRgQ5K>(f_next, hd_next, qs[0], qs[1], qs[2], qs[3]);
    }
    pf_barrier();                                         // (every wave's copies have landed and its reads are through: the slots are free)
    };
    const uint32_t live_tiles = (count + 31U) / 32U;
    if constexpr (TILES == 4U) {
        if (live_tiles >= 4U) run_unit(std::integral_constant<uint32_t, 4>{});
        else if (live_tiles == 3U) run_unit(std::integral_constant<uint32_t, 3>{});
        else if (live_tiles == 2U) run_unit(std::integral_constant<uint32_t, 2>{});
        else run_unit(std::integral_constant<uint32_t, 1>{});
    } else {
        static_assert(TILES == 1U, "live tiles of the four-wave form");
        run_unit(std::integral_constant<uint32_t, 1>{});
    }
    }   // listed units
    }
}

}  // namespace strix950
