// The Q8_0 linear operators: the A8 image of activation rows and the Q8_0 x A8 products. See include/mi355_strix.h for the contract of
// every entry point; reference file:line citations are relative to the reference tree.
#include "a8_rows.hpp"
#include "gemm_q8_0.hpp"

#include <type_traits>

namespace strix950 {

// ======================================================================================================== Q8_0 x A8 GEMV
// One aligned group of 32 lanes per output row: lane l owns the reference's accumulator lane l (groups g = l, l + 32,
// ... ascending), then the tree32 butterfly. Up to RB activation rows share one sweep of the weight row.
// Reference: src/cpu/core/reference.cpp:57-84, src/core/integer_math.hpp:11-13,43-47.
// A block (34 bytes: fp16 scale, 32 codes) is fetched as nine aligned dwords (two 128-bit loads and one 32-bit load) around its codes, wherever the
// 2-byte aligned row starts, and shifted into place; no dword is read that holds no byte of it. (Rows of 4128 and 1056 features by seventeen 16-bit loads a
// block: 8 rows x 8192 outputs 25.8 us, now 23.2, 4 x 4096 9.1, 8.7.) DW: the rows are 4-byte aligned, so the place follows from the block's number (1 row of
// 4096 x 4096 4.5 us, from the address 4.8).
// CHAIN (RB = 1): the row contract of the reference's dense A8 profile (src/hip_q8_rows_gemv.hpp:1155-1170; host statement
// tests/dense_a8_small_reference_tests.cpp:93-104): acc = +0, then for the blocks in ascending order acc = fma(float(d_w) * delta,
// float(dot), acc), and a NaN result is stored as 0x7fc00000. The lanes evaluate their blocks as before and leave every block's
// (scale, dot) pair in LDS; lane 0 of the output's 32 lanes then walks them in order.
constexpr uint32_t kGemvChainMaxGroups = 256;          // in <= 8192 (kDenseA8MaxWidth, src/hip_q8_rows_gemv.hpp:1176)
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
template <int RB, bool DW, bool CHAIN = false>
__global__ __launch_bounds__(256) void gemv_q8_0_a8_kernel(mi355_q8a8_view v) {
    __shared__ float2 chain_pairs[CHAIN ? 8 : 1][CHAIN ? kGemvChainMaxGroups : 1];
    const uint32_t o = blockIdx.x * 8U + (threadIdx.x >> 5), l = threadIdx.x & 31U, row0 = blockIdx.y * RB;
    if (o >= v.count) return;
    const uint32_t groups = v.in / 32U;
    const uint32_t nr = v.rows - row0 < static_cast<uint32_t>(RB) ? v.rows - row0 : static_cast<uint32_t>(RB);
    const uint8_t* wrow = v.weight + static_cast<size_t>(o) * v.row_bytes;
    float lane[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) lane[r] = 0.0F;
    // (unrolled: the loads of four of the lane's groups are in flight together; the accumulation order does not change)
#pragma unroll 4
    for (uint32_t g = l; g < groups; g += 32U) {
        const unsigned short* b = reinterpret_cast<const unsigned short*>(wrow + static_cast<size_t>(g) * kQ80Block);
        const float scale = half_bits_to_float(b[0]);
        int w[8];
        const uint32_t c0 = g * kQ80Block + 2U, shift = (DW ? c0 : static_cast<uint32_t>(reinterpret_cast<uintptr_t>(b + 1))) & 3U;   // first code byte: 0 or 2 past a dword boundary
        const uint32_t* dw = DW ? reinterpret_cast<const uint32_t*>(wrow) + (c0 >> 2) : reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(b + 1) - shift);
        const u32x4_a4 lo4 = *reinterpret_cast<const u32x4_a4*>(dw), hi4 = *reinterpret_cast<const u32x4_a4*>(dw + 4);
        const uint32_t last = dw[shift ? 8 : 7];                          // (an aligned block ends with its eighth dword)
        const uint32_t d[9] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w, last};
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = static_cast<int>(__builtin_amdgcn_alignbyte(d[i + 1], d[i], shift));
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            if (static_cast<uint32_t>(r) < nr) {
                const int4* xc = reinterpret_cast<const int4*>(v.codes + static_cast<size_t>(row0 + r) * v.x_stride + g * 32U);
                const int4 a = xc[0], c = xc[1];
                int dot = 0;
                dot = __builtin_amdgcn_sdot4(w[0], a.x, dot, false); dot = __builtin_amdgcn_sdot4(w[1], a.y, dot, false);
                dot = __builtin_amdgcn_sdot4(w[2], a.z, dot, false); dot = __builtin_amdgcn_sdot4(w[3], a.w, dot, false);
                dot = __builtin_amdgcn_sdot4(w[4], c.x, dot, false); dot = __builtin_amdgcn_sdot4(w[5], c.y, dot, false);
                dot = __builtin_amdgcn_sdot4(w[6], c.z, dot, false); dot = __builtin_amdgcn_sdot4(w[7], c.w, dot, false);
                const float xd = v.deltas[static_cast<size_t>(row0 + r) * (v.x_stride / 32U) + g];
                if constexpr (CHAIN) chain_pairs[threadIdx.x >> 5][g] = make_float2(scale * xd, static_cast<float>(dot));
                else lane[r] = lane[r] + static_cast<float>(dot) * (scale * xd);
            }
        }
    }
    if constexpr (CHAIN) {
        // the pairs were written by lanes of this wave: program order of one wave's LDS accesses
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (l == 0) {
            float acc = 0.0F;
            for (uint32_t g = 0; g < groups; ++g) {
                const float2 c = chain_pairs[threadIdx.x >> 5][g];
                acc = __builtin_fmaf(c.x, c.y, acc);
            }
            v.out[static_cast<size_t>(row0) * v.out_stride + o] = acc != acc ? __builtin_bit_cast(float, 0x7fc00000U) : acc;
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        float p = lane[r];
        p = p + xor16_f(p); p = p + xor8_f(p); p = p + xor4_f(p); p = p + xor2_f(p); p = p + xor1_f(p);
        if (l == 0 && static_cast<uint32_t>(r) < nr) {
            float* y = &v.out[static_cast<size_t>(row0 + r) * v.out_stride + o];
            *y = v.accumulate ? *y + p : p;
        }
    }
}

}  // namespace strix950

using namespace strix950;

namespace {
int32_t a8_image(const A8RowArgs& a, uint32_t kind, uint32_t rows, hipStream_t st) {
    const uint32_t threads = a8_row_threads(a.width);
    if (kind == MI355_INPUT_F32) a8_rows_kernel<0><<<rows, threads, 0, st>>>(a);
    else if (kind == MI355_INPUT_F16) a8_rows_kernel<1><<<rows, threads, 0, st>>>(a);
    else a8_rows_kernel<2><<<rows, threads, 0, st>>>(a);
    STRIX_LAUNCHED("quantize_a8");
    return MI355_OK;
}
int32_t quantize_a8(const void* x, uint32_t kind, uint32_t rows, uint32_t width, uint64_t x_stride, int8_t* codes, float* deltas,
                    int32_t* sums, uint32_t* status, uint32_t status_mode, uint32_t nan_delta, mi355_stream stream) {
    STRIX_REQUIRE(width % 32U == 0, "A8 activation width must be a multiple of 32");
    STRIX_REQUIRE(kind <= MI355_INPUT_BF16, "A8: unknown input kind");
    if (rows == 0 || width == 0) return MI355_OK;
    STRIX_REQUIRE(x && codes && deltas, "A8: null pointer");
    STRIX_REQUIRE(rows <= 65535U, "A8: at most 65535 rows per call");
    const bool vec = aligned(x, 16) && x_stride % 16U == 0 && aligned(codes, 8);
    return a8_image(A8RowArgs{static_cast<const uint8_t*>(x), x_stride, width, codes, deltas, sums, status, status ? status_mode : kA8StatusNone, vec, nan_delta},
                    kind, rows, hs(stream));
}
}  // namespace

extern "C" {

int32_t mi355_quantize_a8(const void* x, uint32_t kind, uint32_t rows, uint32_t width, uint64_t x_stride, int8_t* codes, float* deltas,
                          int32_t* sums, uint32_t* status, mi355_stream stream) {
    return quantize_a8(x, kind, rows, width, x_stride, codes, deltas, sums, status, kA8StatusOr, 0U, stream);
}

int32_t mi355_quantize_a8_fresh(const void* x, uint32_t kind, uint32_t rows, uint32_t width, uint64_t x_stride, int8_t* codes, float* deltas,
                                int32_t* sums, uint32_t* status, mi355_stream stream) {
    return quantize_a8(x, kind, rows, width, x_stride, codes, deltas, sums, status, kA8StatusStore, 0U, stream);
}

int32_t mi355_dense_a8_quantize(const void* x, uint32_t kind, uint32_t rows, uint32_t width, uint64_t x_stride, int8_t* codes, float* deltas,
                                mi355_stream stream) {
    return quantize_a8(x, kind, rows, width, x_stride, codes, deltas, nullptr, nullptr, kA8StatusNone, 1U, stream);
}

int32_t mi355_gemv_q8_0_a8_chain(const mi355_q8a8_view* v, mi355_stream stream) {
    STRIX_REQUIRE(v, "Q8_0 chain product: null view");
    STRIX_REQUIRE(v->in % 64U == 0 && v->in <= 32U * kGemvChainMaxGroups, "Q8_0 chain product: width must be a multiple of 64, at most 8192");   // dense_a8_width, src/hip_q8_rows_gemv.hpp:1184
    STRIX_REQUIRE(!v->accumulate, "Q8_0 chain product: the chain starts at +0 (no accumulate)");
    if (v->rows == 0 || v->count == 0) return MI355_OK;
    STRIX_REQUIRE(v->weight && v->codes && v->deltas && v->out, "Q8_0 chain product: null pointer");
    STRIX_REQUIRE(aligned(v->weight, 4) && v->row_bytes % 4U == 0, "Q8_0 chain product: weight rows must be 4-byte aligned");
    STRIX_REQUIRE(aligned(v->codes, 16) && v->x_stride % 32U == 0 && v->x_stride >= v->in, "Q8_0 chain product: codes must be 16-byte aligned with x_stride a multiple of 32");
    STRIX_REQUIRE(v->row_bytes >= v->in / 32U * kQ80Block && v->out_stride >= v->count && v->rows <= 65535U, "Q8_0 chain product: stride shorter than the row, or too many rows");
    gemv_q8_0_a8_kernel<1, true, true><<<dim3((v->count + 7U) / 8U, v->rows), 256, 0, hs(stream)>>>(*v);
    STRIX_LAUNCHED("gemv_q8_0_a8 chain");
    return MI355_OK;
}

int32_t mi355_gemv_q8_0_a8(const mi355_q8a8_view* v, mi355_stream stream) {
    STRIX_REQUIRE(v, "Q8_0 product: null view");
    STRIX_REQUIRE(v->in % 32U == 0, "Q8_0 product width must be a multiple of 32");
    if (v->rows == 0 || v->count == 0) return MI355_OK;
    STRIX_REQUIRE(v->weight && v->codes && v->deltas && v->out, "Q8_0 product: null pointer");
    STRIX_REQUIRE(aligned(v->weight, 2) && v->row_bytes % 2U == 0, "Q8_0 product: weight rows must be 2-byte aligned");
    STRIX_REQUIRE(aligned(v->codes, 16) && v->x_stride % 32U == 0 && v->x_stride >= v->in, "Q8_0 product: codes must be 16-byte aligned with x_stride a multiple of 32");
    STRIX_REQUIRE(v->row_bytes >= v->in / 32U * kQ80Block && v->out_stride >= v->count, "Q8_0 product: stride shorter than the row");
    const uint32_t grid = (v->count + 7U) / 8U;
    const bool dw = aligned(v->weight, 4) && v->row_bytes % 4U == 0;
    hipStream_t st = hs(stream);
    // up to RB activation rows share one sweep of a weight row; more rows are further blocks of the same launch (grid.y)
    const auto launch = [&](auto rb_constant) {
        constexpr int RB = decltype(rb_constant)::value;
        const dim3 g(grid, (v->rows + RB - 1U) / RB);
        if (dw) gemv_q8_0_a8_kernel<RB, true><<<g, 256, 0, st>>>(*v);
        else gemv_q8_0_a8_kernel<RB, false><<<g, 256, 0, st>>>(*v);
    };
    STRIX_REQUIRE((v->rows + 15U) / 16U <= 65535U, "Q8_0 product: too many rows for one launch");
    // A sweep of few outputs leaves the chip idle, and its time is a workgroup's: rows share one only as far as the launch then still has three workgroups a compute
    // unit (of eight outputs each), four rows up to five (six of rows of 4096 features and more; past eight rows, and past five workgroups, while the weights are few). us, rows a workgroup 1, 2, 4, 8 and tiles:
    //   8192 x 512: 8 rows (512 workgroups of one row) 5.5, 6.9, 9.3, 14.2, 18.9; 16 rows (512 of two) 8.7, 7.6, 9.2, 14.1, 19.0; 64 rows (1024 of four) 28.5, 19.8, 15.7, -, 27.9
    //   2048 x 2048: 3 rows (768 of one) 3.3, 3.6, 3.9; 4 rows (512 of two) 3.8, 3.6, 4.3; 8 rows (512 of four) 5.4, 4.5, 4.5, 5.8, 7.9; 16 rows (1024) -, 6.6, 5.8, 6.0, 8.1;
    //   32 rows (2048) -, 11.1, 9.1, 8.5, 8.2; 6144 x 4096: 8 rows (1024) -, 18.1, 15.3, 19.5, 17.4, 12 rows (1536) -, -, 19.8, 21.4, 17.5; 2048 x 10240: 8 rows (2560) -, -, 13.7, 11.6, 15.3;
    //   5, 8 rows, four | eight: 8192 x 4096 (1024) 18.5, 19.7 | 20.7, 28.1 (tiles 21.9), 8192 x 5120 (1280) 20.6, 22.5 | 21.9, 29.1 (22.3), 2112 x 6019 (1506) 9.1, 10.9 | 8.3, 10.2,
    //   3072 x 6144 (1536) 9.1, 11.3 | 8.9, 11.0, 4096 x 6144 11.1, 13.8 | 11.2, 14.1, 5120 x 6144 14.2, 17.5 | 14.8, 18.8 (16.0)
    // Five to eight rows of many weights are on the matrix cores, whose time hardly depends on the rows but is that of whole rounds of tiles, one to a compute unit: in one round
    // always, in more as far as the last one is full, the more rows the less so, and of rows below 4096 features, whose tiles are mostly start and
    // end, only full ones. 5, 8 rows, sweep of eight | tiles (rounds begun, of which filled): 4096 x 8192 15.0, 18.3 | 14.3 (1, 1); 7168 x 7168 22.6, 28.4 | 22.7
    // (1, 0.88); 6144 x 6144 18.3, 24.0 | 18.2 (1, 0.75); 2048 x 16384 16.7, 20.7 | 16.5 (2, 2); 4096 x 14336 22.2, 27.4 | 25.2 (2, 1.75); 8192 x 12288 35.8, 44.8 | 42.6 (2, 1.5);
    // 8192 x 10240 31.6, 38.8 | 42.0 (2, 1.25); 3072 x 12288 16.8, 20.0 | 23.4 (2, 1.5); 2048 x 28672 23.0, 28.1 | 29.4 (4, 3.5); 1024 x 28672 13.8, 16.6 | 26.3 (4, 3.5).
    const uint64_t known = v->rows == 1U ? 0U : compute_units(), units = known ? known : 1U, weights = static_cast<uint64_t>(v->in) * v->count;
    const auto groups = [&](uint32_t rb) { return static_cast<uint64_t>(grid) * ((v->rows + rb - 1U) / rb); };
    const auto rounds = [&](uint64_t blocks) { return (blocks + units - 1U) / units; };
    const auto few_rows_tiled = [&] {        // of five to eight rows
        const uint64_t tiles = gemm_blocks<8, 1>(v->count, v->rows), places = rounds(tiles) * units;
        if (weights < (7ULL << 22)) return false;
        if (places == units) return true;
        return v->in < 4096U ? v->in >= 2048U && 16U * tiles >= 15U * places : 10U * (places - tiles) <= (v->rows - 5U) * places;
    };
    if (v->rows == 1U || groups(1U) <= 3U * units) launch(std::integral_constant<int, 1>{});
    else if (v->rows == 2U || groups(2U) <= 3U * units) launch(std::integral_constant<int, 2>{});
    else if (v->rows <= 4U || (groups(4U) <= 5U * units && (v->rows <= 8U || weights < (1ULL << 25))) ||
             (v->rows <= 8U && groups(4U) <= 6U * units && v->in >= 4096U && weights < (1ULL << 25))) launch(std::integral_constant<int, 4>{});
    else if (v->rows <= 8U && !few_rows_tiled()) launch(std::integral_constant<int, 8>{});
    else {
        // Tiles of 32 weight x 32 activation rows, 32 x 64 (K split over twice the waves of the last) or 64 x 64, whichever rounds take the shortest: a round is
        // 3.0 + 3.9 n, 3.3 + 6.2 n, 3.5 + 10.2 n us long for n runs of 64 groups a row, and a stripe of tiles stays on one of eight dies (gemm_blocks counts what that leaves empty).
        // us, 32 x 32 | 32 x 64 | 64 x 64 (rounds): 1024, 4096, 8192 features, 96 rows x 4096 13.7, 22.7, 38.6 | 9.3, 17.6, 31.1 | 12.4, 26.2, 46.6 (2, 1, 1); 427 x 2195 26.2, 43.0, 73.6 |
        // 17.2, 31.8, 55.6 | 23.0, 48.8, 89.1 (4, 2, 2); 128 x 6144 20.3, 33.8, 57.3 | 16.8, 32.2, 57.7 | 12.8, 27.3, 50.8 (3, 2, 1); 800 x 1280 26.0, 42.9, 74.6 | 23.4, 44.8, 80.3 | 22.9, 48.7,
        // 89.6 (4, 3, 2). What the tiles do not take stays on the row sweep.
        const uint64_t n = (v->in / 32U + 63U) / 64U;
        const uint64_t narrow = rounds(gemm_blocks<8, 1>(v->count, v->rows)) * (30U + 39U * n), tall = rounds(gemm_blocks<8, 2>(v->count, v->rows)) * (33U + 62U * n),
                       wide = rounds(gemm_blocks<4, 2>(v->count, v->rows)) * (35U + 102U * n);
        const bool taken = v->rows <= 32U || (narrow <= tall && narrow <= wide) ? launch_gemm_q8_0<8, 1>(*v, st)
                           : tall <= wide ? launch_gemm_q8_0<8, 2>(*v, st) : launch_gemm_q8_0<4, 2>(*v, st);
        if (!taken) launch(std::integral_constant<int, 16>{});
    }
    STRIX_LAUNCHED("gemv_q8_0_a8");
    return MI355_OK;
}

}  // extern "C"
