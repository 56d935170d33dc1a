// Routed experts (and a dense FFN as the one-expert case) on the matrix-core sweep of q4k_mma.hpp, for work items of up to 128
// activation rows, 32 outputs a tile.
//   project: the gate tile and the up tile of the same 32 features share the activation rows of a sweep; the values leave through the
//            reference's SwiGLU + A8 re-quantisation of the 32-value group (src/cpu/core/routed_expert.cpp:147-170, :403-427).
//   down:    32 hidden outputs against the A8 image of h (src/cpu/core/routed_expert.cpp:429-447, src/moe_a8_down_contract.cpp:146).
// An item longer than 2 NAL rows is served in chunks; the second and later sweeps of the tile's weights come from the cache.
// dense_rows > 0: no plan, expert 0, assignment i = row i, an "item" is a chunk of 2 NAL rows.
//
// Workgroup (x, y) takes tiles x run .. x run + run - 1 of item y.
#pragma once
#include "plan_layout.hpp"
#include "q4k_mma.hpp"

namespace strix950 {

// What a launch works on beside the weights and rows.
struct MmaLaunch { uint32_t assignments, dense_rows, tiles, run; };
struct MmaArgs { mi355_moe_weights w; RowsK r; MmaLaunch l; };
// The argument block of a kernel whose only argument it is, read again where it is used: the sixty words of the row views are wanted once
// per run of tiles and once per value that leaves, and held in scalar registers over the sweep they push its own out into vector lanes
// (106 spilled, and as many lane reads per tile).
__device__ __forceinline__ const MmaArgs& mma_args() {
    typedef const __attribute__((address_space(4))) MmaArgs args_segment;
    args_segment* p = (args_segment*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const MmaArgs*)p;
}

struct MmaItem { uint32_t e, begin, end; };
__device__ __forceinline__ MmaItem mma_item(const MmaArgs& k, uint32_t width) {
    if (k.l.dense_rows) {                                   // one chunk of the batch per blockIdx.y
        const uint32_t begin = blockIdx.y * width, end = begin + width;
        return {0U, begin, end < k.l.dense_rows ? end : k.l.dense_rows};
    }
    const WorkItem item = work_item(k.w, k.r, plan_items_at(k.w.experts, k.l.assignments), blockIdx.y);
    return {static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(item.e)), static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(item.begin)),
            static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(item.end))};
}
// The rows c0 .. c0 + n of the plan's order (or of a dense batch), as mma_run asks for them; put_addresses(args, a, i) resolves every address
// of row a, assignment i, once, so that nothing else of the kernel does. img: the A8 image the rows are read from. DIRECT: a dense batch
// over one image per row at a stride, which needs no look-up - an instance of its own, because the strides and bases held for it cost
// the planned batches 1.5 % (dense 27648 x 5120, 8 rows: 86.5 -> 84.6 us). PUT: the emitter reads the row table.
template <uint32_t ACTS, bool DIRECT, bool PUT, class Put>
struct MmaRowsOf {
    static constexpr bool kDirect = DIRECT, kPut = PUT;
    static constexpr uint32_t kActs = ACTS;             // rows that the row table has room for
    uint32_t c0;
    const A8Image& img;
    uint32_t dense;
    lds_u64* at;
    lds_u32* slot;
    Put put_addresses;
    __device__ __forceinline__ const uint8_t* codes(uint32_t a) const { return reinterpret_cast<const uint8_t*>(img.codes) + (c0 + a) * img.codes_rs; }
    __device__ __forceinline__ const uint8_t* table(uint32_t a, bool deltas) const {
        const uint8_t* const from = deltas ? reinterpret_cast<const uint8_t*>(img.deltas) : reinterpret_cast<const uint8_t*>(img.sums);
        return from + (c0 + a) * (deltas ? img.deltas_rs : img.sums_rs);
    }
    __device__ __forceinline__ const uint32_t* word(uint32_t a) const {       // (rows that no plan names: any word, of the argument block)
        const MmaArgs& args = mma_args();
        return !dense && !args.r.union_plan ? args.r.plan + plan_order_at(args.w.experts) + c0 + a : &args.l.dense_rows;
    }
    __device__ __forceinline__ void put(uint32_t a, uint32_t n, uint32_t word) const {
        const MmaArgs& args = mma_args();
        const uint32_t position = c0 + (a < n ? a : 0U), i = dense ? position : args.r.union_plan ? union_assignment(args.r.union_plan, position) : word;
        slot[a] = i;
        put_addresses(args, a, i);
    }
};
template <class P> __device__ __forceinline__ uint64_t address(const P* p) { return reinterpret_cast<uint64_t>(p); }

// The sweep of a chunk of n rows, run(NAL): of the wide form with no chain for the result registers past a short chunk.
template <int NAL, bool WIDE, class Run> __device__ __forceinline__ void mma_chunk(uint32_t n, Run run) {
    if constexpr (WIDE) {
        if (n > 24U) run(std::integral_constant<int, 16>{});
        else if (n > 16U) run(std::integral_constant<int, 12>{});
        else if (n > 8U) run(std::integral_constant<int, 8>{});
        else run(std::integral_constant<int, 4>{});
    } else run(std::integral_constant<int, NAL>{});
}

// Waves per SIMD: what the LDS of a workgroup allows (four of 36 KB, three of 44 or 46 KB, two of eight wavefronts and 73 KB), which for 16 rows the compiler misses
// by a few registers when it is not told (200 rows of hidden 2048 / ffn 768 / 128 experts: 192.8 -> 172.3 us a layer, 219.6 before the run).
template <int FMT, int NAL, int DEPTH, bool DIRECT, bool WIDE>
__global__ __launch_bounds__(WIDE ? 512 : 256, NAL == 2 || WIDE ? 4 : NAL <= 8 ? 3 : 2) void q4k_mma_project_kernel(MmaArgs k) {
    constexpr uint32_t ACTS = mma_acts<NAL>();
    __shared__ __attribute__((aligned(16))) uint8_t ring_mem[mma_ring_bytes<FMT, NAL, 2, DEPTH, 1>()];
    __shared__ float red_mem[mma_reduce_floats<NAL, 2>()];
    __shared__ uint64_t at_mem[mma_row_words<NAL, 3>()];
    __shared__ uint32_t slot_mem[ACTS];
    lds_u64* const at = (lds_u64*)at_mem;
    lds_u32* const slot = (lds_u32*)slot_mem;
    const MmaItem item = mma_item(k, ACTS);
    if (item.begin == item.end) return;
    const uint32_t tile0 = blockIdx.x * k.l.run, tiles = k.l.tiles - tile0 < k.l.run ? k.l.tiles - tile0 : k.l.run;
    const size_t base = static_cast<size_t>(item.e) * k.w.gate_expert_stride + static_cast<size_t>(tile0 * 32U) * k.w.gate_row_stride;
    const uint8_t* const wrows[2] = {k.w.gate + base, k.w.up + base};
    for (uint32_t c0 = item.begin; c0 < item.end; c0 += ACTS) {
        const uint32_t n = item.end - c0 < ACTS ? item.end - c0 : ACTS;
        const auto put = [&](const MmaArgs& args, uint32_t a, uint32_t i) {
            const RowsK& r = args.r;
            const uint32_t row = r.row_of(i);
            at[a] = address(r.in.codes_of(row));
            at[ACTS + a] = address(r.in.deltas_of(row));
            at[2U * ACTS + a] = address(r.in.sums_of(row));
            if (!r.h.codes) return;
            at[3U * ACTS + a] = address(r.h_codes_of(i));
            at[4U * ACTS + a] = address(r.h_deltas_of(i));
            at[5U * ACTS + a] = address(r.h_sums_of(i));
        };
        const MmaRowsOf<ACTS, DIRECT, true, decltype(put)> rows{c0, k.r.in, k.l.dense_rows, at, slot, put};
        const auto emit = [&](uint32_t tile, uint32_t v, uint32_t lane, const float (&value)[2]) {
            const uint32_t j = lane & 31U, h = lane >> 5;
            const MmaArgs& args = mma_args();
            const RowsK& r = args.r;
            // lane (feature j, half h) holds gate and up of activation row 2v + h; a half past the chunk computes on and stores nothing
            const bool live = 2U * v + h < n;
            const uint32_t a = live ? 2U * v + h : 0U, grp = tile0 + tile, at_out = grp * 32U + j;
            const float g = value[0], u = value[1];
            float gc = g, uc = u;
            swiglu_clamp(gc, uc, args.w.swiglu_limit);
            const float hv = (gc / (1.0F + exp_of(args.w.exp_kind, -gc))) * uc;
            if (live && (r.gate_out || r.up_out || r.h_out)) {
                const uint32_t i = slot[a];
                if (r.gate_out) r.inter_of(r.gate_out, i)[at_out] = g;
                if (r.up_out) r.inter_of(r.up_out, i)[at_out] = u;
                if (r.h_out) r.inter_of(r.h_out, i)[at_out] = hv;
            }
            if (!r.h.codes) return;             // projection only (the probe form): no A8 image of h
            const uint64_t votes = __ballot(!(finite_f(g) && finite_f(u) && finite_f(hv)));
            const float amax = max32(__builtin_fabsf(hv));
            const bool tiny = amax > 0.0F && amax < 0x1p-119F;
            const float dl = (amax == 0.0F || tiny) ? 1.0F : amax / 127.0F;
            const int code = a8_code(hv, dl, tiny);
            const int sum = sum32_i(code);
            if (!live) return;
            if (h ? votes >> 32 : votes & 0xffffffffULL) {
                if (j == 0) {
                    atomicOr(r.status_of(r.row_of(slot[a])), r.nonfinite_bit);
                    atomicOr(r.job_status, static_cast<uint32_t>(MI355_STATUS_NONFINITE_PROJECTION));
                }
                return;
            }
            reinterpret_cast<int8_t*>(at[3U * ACTS + a])[at_out] = static_cast<int8_t>(code);
            if (j == 0) {
                reinterpret_cast<float*>(at[4U * ACTS + a])[grp] = dl;
                reinterpret_cast<int32_t*>(at[5U * ACTS + a])[grp] = sum;
            }
        };
        const auto run = [&](auto nal) __attribute__((always_inline)) {
            mma_run<FMT, decltype(nal)::value, DEPTH, 1, 2, true, WIDE>((lds_u8*)ring_mem, nullptr, (lds_f32*)red_mem, wrows, k.w.gate_row_stride, k.w.hidden / 256U, tiles, kMmaRows, n, rows, emit);
        };
        mma_chunk<NAL, WIDE>(n, run);
    }
}

// GATE_UP: the same sweep over gate (blockIdx.z = 0) or up (1) rows against the input image, raw values out to the gate / up
// intermediates - the dense FFN's projection when that workspace exists (two launches' worth of narrow workgroups fill the
// compute units better than the fused form's wide ones: 27648 x 5120, 8 rows: 54 + 5 us against 70 us).
template <int FMT, int NAL, int DEPTH, int TEAMS, bool DIRECT, bool GATE_UP = false>
__global__ __launch_bounds__(NAL == 16 ? 512 : 256 * TEAMS, NAL == 16 ? 4 : 1) void q4k_mma_down_kernel(MmaArgs k) {
    // the wide form: over two tiles at a time, as if they were of two matrices
    constexpr uint32_t ACTS = mma_acts<NAL>(), NM = mma_wide<FMT, NAL>() ? 2U : 1U, TILE = NM * kMmaRows;
    __shared__ __attribute__((aligned(16))) uint8_t ring_mem[mma_ring_bytes<FMT, NAL, NM, DEPTH, TEAMS>()];
    __shared__ float xbuf_mem[mma_exchange_floats<NAL, TEAMS>()];
    __shared__ float red_mem[mma_reduce_floats<NAL, NM>()];
    __shared__ uint64_t at_mem[mma_row_words<NAL, 1>()];
    __shared__ uint32_t slot_mem[ACTS];
    lds_u64* const at = (lds_u64*)at_mem;
    lds_u32* const slot = (lds_u32*)slot_mem;
    if (!GATE_UP && (*k.r.job_status & MI355_STATUS_NONFINITE_PROJECTION)) return;
    const uint8_t* const matrix = GATE_UP ? (blockIdx.z ? k.w.up : k.w.gate) : k.w.down;
    const uint64_t expert_stride = GATE_UP ? k.w.gate_expert_stride : k.w.down_expert_stride, row_stride = GATE_UP ? k.w.gate_row_stride : k.w.down_row_stride;
    const MmaItem item = mma_item(k, ACTS);
    if (item.begin == item.end) return;
    const uint32_t tile0 = blockIdx.x * k.l.run, tiles = k.l.tiles - tile0 < k.l.run ? k.l.tiles - tile0 : k.l.run;
    const uint8_t* wrows[NM];
#pragma unroll
    for (uint32_t m = 0; m < NM; ++m) wrows[m] = matrix + static_cast<size_t>(item.e) * expert_stride + static_cast<size_t>(tile0 * TILE + m * kMmaRows) * row_stride;
    for (uint32_t c0 = item.begin; c0 < item.end; c0 += ACTS) {
        const uint32_t n = item.end - c0 < ACTS ? item.end - c0 : ACTS;
        const auto put = [&](const MmaArgs& args, uint32_t a, uint32_t i) {
            const RowsK& r = args.r;
            const A8Image& img = GATE_UP ? r.in : r.h;
            const uint32_t from = GATE_UP ? r.row_of(i) : i;
            at[a] = address(img.codes_of(from));
            at[ACTS + a] = address(img.deltas_of(from));
            at[2U * ACTS + a] = address(img.sums_of(from));
            at[3U * ACTS + a] = GATE_UP ? address(r.inter_of(blockIdx.z ? r.up_out : r.gate_out, i)) : address(r.rawdots_of(i, args.w.hidden));
        };
        const MmaRowsOf<ACTS, DIRECT, !DIRECT, decltype(put)> rows{c0, GATE_UP ? k.r.in : k.r.h, k.l.dense_rows, at, slot, put};
        const auto emit = [&](uint32_t tile, uint32_t v, uint32_t lane, const float (&value)[NM]) {
            const uint32_t a = 2U * v + (lane >> 5), at_out = (tile0 + tile) * TILE + (lane & 31U);
            if (a >= n) return;
            // (the rows of a dense batch: assignment = row, at a stride; the argument block read again at a workgroup's end is one way to memory more)
            float* const out = !DIRECT ? reinterpret_cast<float*>(at[3U * ACTS + a])
                               : GATE_UP ? k.r.inter_of(blockIdx.z ? k.r.up_out : k.r.gate_out, c0 + a) : k.r.rawdots_of(c0 + a, k.w.hidden);
#pragma unroll
            for (uint32_t m = 0; m < NM; ++m) {
                out[at_out + m * kMmaRows] = value[m];
                if (!GATE_UP && k.r.top1_form)      // (top-1: assignment = row)
                    (DIRECT ? k.r : mma_args().r).publish_top1(DIRECT ? c0 + a : slot[a], at_out + m * kMmaRows, value[m]);
            }
        };
        const auto run = [&](auto nal) __attribute__((always_inline)) {
            mma_run<FMT, decltype(nal)::value, DEPTH, TEAMS, NM, TEAMS == 1 && !GATE_UP, mma_wide<FMT, NAL>()>((lds_u8*)ring_mem, (lds_f32*)xbuf_mem, (lds_f32*)red_mem, wrows, row_stride,
                                                                                                  (GATE_UP ? k.w.hidden : k.w.ffn) / 256U, tiles, TILE, n, rows, emit);
        };
        mma_chunk<NAL, mma_wide<FMT, NAL>()>(n, run);
    }
}

}  // namespace strix950
