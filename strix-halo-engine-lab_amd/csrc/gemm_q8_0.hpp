// Q8_0 x A8 products of many activation rows: the exact 32-element group dots on the int8 matrix cores, the reference's fp32 order on
// the vector ALU. out[a][o] = tree32 of 32 lane sums; lane l sums float(dot(g)) * (scale(o, g) * delta(a, g)) over the groups g = l,
// l + 32, ... in ascending order (src/cpu/core/reference.cpp:57-84, src/core/integer_math.hpp:11-13,43-47).
//
// A workgroup of eight waves owns 32 OG weight rows x 32 NA activation rows. KS of its waves split K by lane: wave w takes the lanes
// l = w (mod KS), which are a whole subtree of tree32, so the waves meet only at its last log2(KS) levels (through LDS, once). A wave
// walks its 32 / KS lanes in bit-reversed order and folds a finished lane sum into the partial tree at once - a binary counter, so it
// holds log2(32 / KS) + 1 sums per output and not 32. Per (32 x 32 outputs, group): one v_mfma_i32_32x32x32_i8 started from the bits of
// 1.5 * 2^23, so that its result read as a float is 1.5 * 2^23 + dot and one subtraction makes the dot a float (a conversion costs
// twice an add); the factors scale * delta of two such tiles are one v_mfma_f32_32x32x1_2b_f32 (products rounded once, +0 added); then
// a multiply and an add. Bound by those three vector operations and the two matrix operations they wait for.
// Memory: per stage the KS groups of one lane class in two chunks of 32 groups, for every row of the tile: a thread copies one weight
// block (nine dwords around its 34 bytes, shifted into place; 777 rows of 3104 x 5000, rows aligned to 2 bytes, 133 us by 16-bit loads, 118) and one or two activation groups through registers into one of two LDS
// buffers while the other is multiplied; rows are pitched by 16 bytes so that eight neighbouring rows read different banks.
// What bounds it now, at 4096 x 4096 and 64 x 64 tiles: a stage takes 0.8 us of products (two waves per SIMD, 192 full-rate vector
// operations and six matrix operations each) and 0.4 us of copies that are not hidden; every workgroup pays about 5 us of start and end.
// With every copy from the first cache 1000 rows of 8192 x 16384 take 743 us, where all waves wrote their copies at once 874, now 775; the vector operations alone are 460. A chain whose products and
// operands were asked for a tile ahead (the factors as one v_mfma_f32_32x32x2_f32 a tile, twice the matrix time) waited less and issued no more: 967 us.
// Copying global -> LDS without registers, four stages ahead (raw 34-byte blocks, shifted by the readers) measured 64 us at 500 rows
// against 56: the readers' 32-bit LDS reads cost more than the copies they hide.
// Measured, 4096 x 4096: 500 rows 323 -> 50 us, 1000 rows 640 -> 98 us, 32 rows 31 -> 12 us against the row sweep (gemv_q8_0_a8_kernel).
#pragma once
#include "device_math.hpp"
#include "host_common.hpp"

namespace strix950 {

typedef int32_t mm_i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t mm_i32x16 __attribute__((ext_vector_type(16)));
typedef float mm_f32x32 __attribute__((ext_vector_type(32)));
typedef uint32_t mm_u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr uint32_t kGemmThreads = 512;
template <int KS> constexpr uint32_t gemm_groups() { return 2U * KS; }                        // groups of a stage
template <int KS> constexpr uint32_t gemm_pitch() { return 32U * gemm_groups<KS>() + 16U; }   // bytes of a tile row in LDS
template <int KS> constexpr uint32_t gemm_out_rows() { return 32U * (8U / KS); }

// the value of the stage-pass p of R in lane order: p with its log2(R) bits reversed
template <int R> __device__ __forceinline__ uint32_t gemm_lane_of_pass(uint32_t p) { return __builtin_bitreverse32(p) >> (R == 8 ? 29 : 30); }

template <int KS, int NA>
__global__ __launch_bounds__(kGemmThreads, 2) void gemm_q8_0_a8_kernel(mi355_q8a8_view v, uint32_t o_tiles, uint32_t a_tiles) {
    constexpr uint32_t OT = gemm_out_rows<KS>(), AT = 32U * NA, G = gemm_groups<KS>(), P = gemm_pitch<KS>(), R = 32U / KS;
    constexpr uint32_t LEVELS = R == 8U ? 3U : 2U, ABLK = AT * G / kGemmThreads > 0U ? AT * G / kGemmThreads : 1U;
    static_assert(OT * G == kGemmThreads, "one weight block per thread and stage");
    __shared__ __attribute__((aligned(16))) uint8_t wbuf[2][OT * P];
    __shared__ __attribute__((aligned(16))) uint8_t abuf[2][AT * P];
    __shared__ float wscale[2][G * OT];
    __shared__ float adelta[2][G * AT];
    // tiles of one weight stripe stay on one die (workgroups go to the eight dies in turn): its activation tiles follow each other there
    const uint32_t die = blockIdx.x & 7U, slot = blockIdx.x >> 3, ot = die + 8U * (slot / a_tiles), at = slot % a_tiles;
    if (ot >= o_tiles) return;
    const uint32_t t = threadIdx.x, lane = t & 63U, j = lane & 31U, h = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6), kw = wave % KS, og = wave / KS;
    // The next stage's copies go to LDS in front of a stage's products, a stage after they were asked for, in the first four waves, and behind them, half as long
    // after, in the other four: a SIMD has one wave of each, so that one writes its copies while the other multiplies. All waves behind (tiles of 64 weight
    // rows) or in front (32) -> now: 4096 x 4096, 500 rows 55 -> 50 us, 1000 rows 110 -> 98, 50 rows 18.4 -> 16.6; 100 rows of 8192 x 1024 30.9 -> 27.9; 300 rows of 4096 x
    // 2048 34.3 -> 31.2.
    const bool early = wave < 4U;
    const uint32_t groups = v.in / 32U, chunks = (groups + 31U) / 32U, per_pass = (chunks + 1U) / 2U, stages = R * per_pass;

    // ---- loader role
    const uint32_t wrow = t / G, wg = t % G;
    const uint32_t orow = ot * OT + wrow < v.count ? ot * OT + wrow : v.count - 1U;
    const uint8_t* wsrc = v.weight + static_cast<size_t>(orow) * v.row_bytes;
    const bool loads_acts = t < AT * G;
    const int8_t* asrc[ABLK];
    const float* dsrc[ABLK];
    uint32_t arow[ABLK];
#pragma unroll
    for (uint32_t b = 0; b < ABLK; ++b) {
        arow[b] = (t / G + b * (kGemmThreads / G)) % AT;
        const uint32_t a = at * AT + arow[b] < v.rows ? at * AT + arow[b] : v.rows - 1U;
        asrc[b] = v.codes + static_cast<size_t>(a) * v.x_stride;
        dsrc[b] = v.deltas + static_cast<size_t>(a) * (v.x_stride / 32U);
    }
    uint32_t wd[9], code_shift = 0;
    u32x4 ac[ABLK][2];
    uint32_t scale_next = 0;
    float delta_next[ABLK];
    bool live = false;                               // the stage's group exists
    const auto group_of = [&](uint32_t s) {          // the group this thread copies in stage s
        const uint32_t p = s / per_pass, c = 2U * (s - p * per_pass) + wg / KS;
        return 32U * c + KS * gemm_lane_of_pass<R>(p) + wg % KS;
    };
    const auto fetch = [&](uint32_t s) {
        const uint32_t g = group_of(s), gg = g < groups ? g : groups - 1U;
        const unsigned short* b = reinterpret_cast<const unsigned short*>(wsrc + static_cast<size_t>(gg) * kQ80Block);
        // (nothing here touches a loaded value: the loads are in flight while the previous stage is multiplied)
        scale_next = b[0];
        live = g < groups;
        // the nine aligned dwords around the 32 codes (of an aligned block, and of what ends the tensor, none that holds no byte of the block)
        // (found from the pointer: an address made of an integer would be loaded through the flat path, which the LDS waits wait for as well)
        code_shift = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(b + 1)) & 3U;     // first code byte: 0 or 2 past a dword boundary
        const uint32_t* dw = reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(b + 1) - code_shift);
        const mm_u32x4_a4 lo = *reinterpret_cast<const mm_u32x4_a4*>(dw), hi = *reinterpret_cast<const mm_u32x4_a4*>(dw + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) { wd[i] = lo[i]; wd[4 + i] = hi[i]; }
        wd[8] = dw[code_shift ? 8 : 7];
        if (loads_acts) {
#pragma unroll
            for (uint32_t b2 = 0; b2 < ABLK; ++b2) {
                const u32x4* src = reinterpret_cast<const u32x4*>(asrc[b2] + 32U * gg);
                ac[b2][0] = src[0]; ac[b2][1] = src[1];
                delta_next[b2] = dsrc[b2][gg];
            }
        }
    };
    const auto stage = [&](uint32_t buf) {
        u32x4 w0, w1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            w0[i] = __builtin_amdgcn_alignbyte(wd[i + 1], wd[i], code_shift);
            w1[i] = __builtin_amdgcn_alignbyte(wd[i + 5], wd[i + 4], code_shift);
        }
        u32x4* wdst = reinterpret_cast<u32x4*>(&wbuf[buf][wrow * P + 32U * wg]);
        wdst[0] = w0; wdst[1] = w1;
        // a group past the row: factor 0 * 0 and finite codes, which adds +0 to a sum that never is -0
        wscale[buf][wg * OT + wrow] = live ? half_bits_to_float(scale_next) : 0.0F;
        if (loads_acts) {
#pragma unroll
            for (uint32_t b = 0; b < ABLK; ++b) {
                u32x4* adst = reinterpret_cast<u32x4*>(&abuf[buf][arow[b] * P + 32U * wg]);
                adst[0] = ac[b][0]; adst[1] = ac[b][1];
                adelta[buf][wg * AT + arow[b]] = live ? delta_next[b] : 0.0F;
            }
        }
    };

    float bias = 12582912.0F;
    asm("" : "+v"(bias));
    mm_i32x16 magic;
#pragma unroll
    for (int i = 0; i < 16; ++i) magic[i] = 0x4B400000;
    asm("" : "+v"(magic));          // kept in registers: as a known constant it would be written again in front of every product
    float acc[NA][16], part[LEVELS][NA][16];
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[n][i] = 0.0F;

    const auto tile_terms = [&](uint32_t buf, uint32_t g, int n, const mm_f32x32& factors, int first) {
        const uint8_t* wp = &wbuf[buf][(32U * og + j) * P + 32U * g + 16U * h];
        const uint8_t* ap = &abuf[buf][(32U * n + j) * P + 32U * g + 16U * h];
        const mm_i32x4 b = *reinterpret_cast<const mm_i32x4*>(wp), a = *reinterpret_cast<const mm_i32x4*>(ap);
        const mm_i32x16 dot = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, magic, 0, 0, 0);
        float d[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) { const int32_t biased = dot[i]; d[i] = __builtin_bit_cast(float, biased) - bias; }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) d[i] = d[i] * factors[first + i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[n][i] = acc[n][i] + d[i];
    };

    fetch(0);
    stage(0);
    if (early) fetch(1);                                        // (R stages at least)
    __syncthreads();
    uint32_t in_pass = 0, pass = 0;
    for (uint32_t s = 0; s < stages; ++s) {
        const uint32_t buf = s & 1U;
        if (early && s + 1U < stages) stage(buf ^ 1U);
        if (s + (early ? 2U : 1U) < stages) fetch(s + (early ? 2U : 1U));
        const bool second = 2U * in_pass + 1U < chunks;         // the stage's second chunk exists
        const mm_f32x32 none = {0};
        if constexpr (NA == 2) {                                // one factor product per group: its two blocks are the two activation tiles
#pragma unroll
            for (uint32_t c = 0; c < 2U; ++c) {
                if (c == 1U && !second) break;
                const uint32_t g = c * KS + kw;
                const mm_f32x32 f = __builtin_amdgcn_mfma_f32_32x32x1f32(adelta[buf][g * AT + lane], wscale[buf][g * OT + 32U * og + j], none, 0, 0, 0);
                tile_terms(buf, g, 0, f, 0);
                tile_terms(buf, g, NA - 1, f, 16);
            }
        } else {                                                // its two blocks are the groups of the two chunks
            const uint32_t g = h * KS + kw;
            const mm_f32x32 f = __builtin_amdgcn_mfma_f32_32x32x1f32(adelta[buf][g * AT + j], wscale[buf][g * OT + 32U * og + j], none, 0, 0, 0);
            tile_terms(buf, kw, 0, f, 0);
            if (second) tile_terms(buf, KS + kw, 0, f, 16);
        }
        if (++in_pass == per_pass) {                            // the lane sum is complete: fold it into the partial tree
            in_pass = 0;
            const uint32_t p = pass++;
            const auto each = [&](auto f) {
#pragma unroll
                for (int n = 0; n < NA; ++n)
#pragma unroll
                    for (int i = 0; i < 16; ++i) f(n, i);
            };
            if ((p & 1U) == 0U) each([&](int n, int i) { part[0][n][i] = acc[n][i]; acc[n][i] = 0.0F; });
            else {
                each([&](int n, int i) { acc[n][i] = part[0][n][i] + acc[n][i]; });
                if ((p & 2U) == 0U) each([&](int n, int i) { part[1][n][i] = acc[n][i]; acc[n][i] = 0.0F; });
                else {
                    each([&](int n, int i) { acc[n][i] = part[1][n][i] + acc[n][i]; });
                    if constexpr (LEVELS == 3U) {
                        if ((p & 4U) == 0U) each([&](int n, int i) { part[2][n][i] = acc[n][i]; acc[n][i] = 0.0F; });
                        else each([&](int n, int i) { acc[n][i] = part[2][n][i] + acc[n][i]; });
                    }
                }
            }
        }
        if (!early && s + 1U < stages) stage(buf ^ 1U);
        __syncthreads();
    }

    // the last levels of the tree across the KS waves: wave kw adds and stores the result registers i = kw (mod KS), one tile at a time
    float* red = reinterpret_cast<float*>(&wbuf[0][0]);
    static_assert(sizeof(wbuf) >= 8U * 16U * 64U * 4U, "reduction space of one tile per wave");
#pragma unroll
    for (int n = 0; n < NA; ++n) {
#pragma unroll
        for (int i = 0; i < 16; ++i) red[(wave * 16U + i) * 64U + lane] = acc[n][i];
        __syncthreads();
#pragma unroll
        for (uint32_t q = 0; q < 16U / KS; ++q) {
            const uint32_t i = q * KS + kw;
            float x[KS];
#pragma unroll
            for (uint32_t w = 0; w < KS; ++w) x[w] = red[((og * KS + w) * 16U + i) * 64U + lane];
#pragma unroll
            for (uint32_t d = KS / 2U; d; d >>= 1)
#pragma unroll
                for (uint32_t w = 0; w < d; ++w) x[w] = x[w] + x[w + d];
            const uint32_t a = at * AT + 32U * n + 8U * (i >> 2) + 4U * h + (i & 3U), o = ot * OT + 32U * og + j;
            if (a < v.rows && o < v.count) {
                float* y = &v.out[static_cast<size_t>(a) * v.out_stride + o];
                *y = v.accumulate ? *y + x[0] : x[0];
            }
        }
        __syncthreads();
    }
}

// Workgroups of a product, and whether the tiles take it: an empty reduction has no group for the loaders to fetch, and a launch counts its
// threads in 32 bits, which tiles of 64 x 64 outputs reach at 2^35 outputs (the row sweep's second grid dimension goes on from there).
template <int KS, int NA>
constexpr uint64_t gemm_blocks(uint32_t count, uint32_t rows) {
    return (static_cast<uint64_t>(count) + 8U * gemm_out_rows<KS>() - 1U) / (8U * gemm_out_rows<KS>()) * 8U * ((rows + 32U * NA - 1U) / (32U * NA));
}
template <int KS, int NA>
constexpr bool gemm_takes(uint32_t in, uint32_t count, uint32_t rows) { return in != 0U && gemm_blocks<KS, NA>(count, rows) * kGemmThreads <= 0xffffffffULL; }
static_assert(!gemm_takes<8, 1>(0U, 70U, 9U) && !gemm_takes<4, 2>(0U, 70U, 4096U) && gemm_takes<4, 2>(32U, 16384U, 65536U));
static_assert(gemm_takes<4, 2>(32U, 32768U, 1048512U) && !gemm_takes<4, 2>(32U, 32768U, 1048560U) && !gemm_takes<4, 2>(32U, 1U << 27, 4096U * 64U));

// false: the row sweep serves the product
template <int KS, int NA>
inline bool launch_gemm_q8_0(const mi355_q8a8_view& v, hipStream_t st) {
    if (!gemm_takes<KS, NA>(v.in, v.count, v.rows)) return false;
    const uint32_t o_tiles = (v.count + gemm_out_rows<KS>() - 1U) / gemm_out_rows<KS>(), a_tiles = (v.rows + 32U * NA - 1U) / (32U * NA);
    const uint32_t blocks = static_cast<uint32_t>(gemm_blocks<KS, NA>(v.count, v.rows));
    gemm_q8_0_a8_kernel<KS, NA><<<blocks, kGemmThreads, 0, st>>>(v, o_tiles, a_tiles);
    return true;
}

}  // namespace strix950
