// Early routes for decode batches: the expert choice leaves the critical path of the layer.
//
// The reference's logits are one ascending fma chain per (row, expert) - `hidden` dependent operations, microseconds of
// latency during which nothing else of the layer can start. The expert *ids* do not need those bits: a dot product in any
// summation order picks the same top-k except where two logits lie within rounding of each other. So the layer runs as
//   1. front launch (layer_front_kernel): early blocks compute the logits as lane-parallel sums (one wave per row and four
//      experts, operands straight into registers) and pick the top-k, the A8 prologue rides beside them, projection blocks
//      sweep gate / up on the early ids as soon as those are tagged, and side blocks run the exact router (the chain, the
//      softmax, the selection, the weights - the reference's bits, written to the caller's ids / weights / scores); the side
//      block that finishes a row compares its exact ids with the early ones and, where they differ, waits for that
//      assignment's speculative waves and repairs the assignment (a copy of the h image the row already holds under another
//      slot, or a sweep on the exact expert) and writes the work items with the exact experts;
//   2. down rows + combine on work items that are exact by then.
// Every output is the exact router's; the early choice only decides which weights stream first.
// Reference (the bits kept): tests/hip_moe_route_launcher_tests.hip:281-330, include/strix/moe/route_policy.hpp:99-156.
#pragma once
#include "route_wave.hpp"
#include "q4k_rows.hpp"

namespace strix950 {

constexpr uint32_t kEarlyExperts = 4;         // experts per early block
constexpr uint32_t kEarlySpinLimit = 1U << 20;      // polls of the selecting block (cannot run out, short of a lost launch)

// ---------------------------------------------------------------------------------------------------- early logits
// Lane l owns features 8 l .. 8 l + 7 of every run of 512; four runs are requested together (36 loads in flight).
template <int KIND>
__device__ __forceinline__ void early_logits_block(const RouteArgs& a, uint32_t row, uint32_t e0, uint32_t epoch) {
    const uint32_t lane = threadIdx.x & 63U;
    float acc[kEarlyExperts];
    const float* wrow[kEarlyExperts];
#pragma unroll
    for (uint32_t i = 0; i < kEarlyExperts; ++i) {
        acc[i] = 0.0F;
        const uint32_t e = e0 + i < a.p.experts ? e0 + i : a.p.experts - 1U;
        wrow[i] = a.wr + static_cast<size_t>(e) * a.hidden;
    }
    const uint8_t* xrow = a.x + row * a.x_stride;
    for (uint32_t k0 = 0; k0 < a.hidden; k0 += 2048U) {
        f32x4 wv[4][kEarlyExperts][2];
        u32x4 xr[4][2];
        bool ok[4];
#pragma unroll
        for (uint32_t s = 0; s < 4U; ++s) {
            const uint32_t k = k0 + 512U * s + 8U * lane;
            ok[s] = k < a.hidden;
            const uint32_t kk = ok[s] ? k : 0U;
#pragma unroll
            for (uint32_t i = 0; i < kEarlyExperts; ++i) {
                wv[s][i][0] = *reinterpret_cast<const f32x4*>(wrow[i] + kk);
                wv[s][i][1] = *reinterpret_cast<const f32x4*>(wrow[i] + kk + 4U);
            }
            if constexpr (KIND == 0) {
                xr[s][0] = *reinterpret_cast<const u32x4*>(xrow + 4U * kk);
                xr[s][1] = *reinterpret_cast<const u32x4*>(xrow + 4U * kk + 16U);
            } else {
                xr[s][0] = *reinterpret_cast<const u32x4*>(xrow + 2U * kk);
            }
        }
#pragma unroll
        for (uint32_t s = 0; s < 4U; ++s) {
            float f[8];
            if constexpr (KIND == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) { f[q] = f_of(xr[s][0][q]); f[4 + q] = f_of(xr[s][1][q]); }
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t h = xr[s][0][q];
                    if constexpr (KIND == 1) { f[2 * q] = half_bits_to_float(h & 0xffffU); f[2 * q + 1] = half_bits_to_float(h >> 16); }
                    else { f[2 * q] = f_of(h << 16); f[2 * q + 1] = f_of(h & 0xffff0000U); }
                }
            }
            if (!ok[s]) {
#pragma unroll
                for (int q = 0; q < 8; ++q) f[q] = 0.0F;
            }
#pragma unroll
            for (uint32_t i = 0; i < kEarlyExperts; ++i) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    acc[i] = __builtin_fmaf(f[q], wv[s][i][0][q], acc[i]);
                    acc[i] = __builtin_fmaf(f[4 + q], wv[s][i][1][q], acc[i]);
                }
            }
        }
    }
    // a logit travels as one 64-bit word {this call's epoch, its bits}: the row's selecting block reads the words until all carry the
    // epoch - no count, no wait for an acknowledgement in between
    unsigned long long* out = reinterpret_cast<unsigned long long*>(a.early_logits) + static_cast<size_t>(row) * (a.early_stride / 2U);
#pragma unroll
    for (uint32_t i = 0; i < kEarlyExperts; ++i) {
        float v = acc[i];
        v = v + xor1_f(v); v = v + xor2_f(v); v = v + xor4_f(v); v = v + xor8_f(v); v = v + xor16_f(v);
        v = v + __shfl_xor(v, 32);
        const uint32_t e = e0 + i;
        if (lane == i && e < a.p.experts) {
            if (a.bias) v = v + a.bias[e];
            // test knob: displaces the early logits (never the exact ones), so that early and exact ids differ
            if (a.early_perturb) v = v + static_cast<float>(a.early_perturb) * 1e-3F * (static_cast<float>((e * 2654435761U) >> 28) - 8.0F);
            __hip_atomic_store(out + e, (static_cast<unsigned long long>(epoch) << 32) | b_of(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// ---------------------------------------------------------------------------------------------------- hand-off between workgroups
// The launches of this file exchange a few words between workgroups: logits, a per-row arrival count, per-assignment counts.
// All of them are read and written by device-scope atomic operations only (they are performed at the memory side, past the
// per-XCD caches), so no cache write-back or invalidation is needed around them: a producer waits until its stores have been
// acknowledged and then counts itself in; the consumer's reads follow its own count operation in program order. Each row's
// count sits in a 128-byte line of its own (32 workgroups counting into one line cost about 0.3 us; all rows' counts in one
// line were measured at 3 us).
__device__ __forceinline__ void stores_acknowledged() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// true in every lane of the one-wave workgroup that arrives last of `parties`; that workgroup leaves the count zero again
__device__ __forceinline__ bool arrive_last(uint32_t* count, uint32_t parties) {
    stores_acknowledged();
    uint32_t seen = 0;
    if ((threadIdx.x & 63U) == 0) seen = __hip_atomic_fetch_add(count, 1U, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    seen = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(seen)));
    asm volatile("" ::: "memory");
    if (seen != parties - 1U) return false;
    if ((threadIdx.x & 63U) == 0) __hip_atomic_store(count, 0U, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// top-k of one row's early logits: greater logit first, lower id on ties. Returns, in lane k < top_k, the expert of slot k.
// A pass = one wave-wide maximum of 32-bit keys (the logit's bits made order preserving) by DPP row shifts and broadcasts, then
// the lowest id among the lanes that hold it.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t max_step_u32(uint32_t v) {
    const uint32_t o = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROW_MASK, 0xF, false));
    return o > v ? o : v;
}
__device__ __forceinline__ uint32_t max_wave_u32(uint32_t v) {
    v = max_step_u32<0x111, 0xF>(v); v = max_step_u32<0x112, 0xF>(v); v = max_step_u32<0x114, 0xF>(v); v = max_step_u32<0x118, 0xF>(v);
    v = max_step_u32<0x142, 0xA>(v); v = max_step_u32<0x143, 0xC>(v);
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}
// ok (all lanes): every logit of the row arrived within the bounded wait.
template <uint32_t PER>
__device__ __forceinline__ uint32_t early_select_row_per(const RouteArgs& a, uint32_t row, uint32_t epoch, bool& ok) {
    const uint32_t lane = threadIdx.x & 63U, E = a.p.experts, K = a.p.top_k;
    const unsigned long long* z = reinterpret_cast<const unsigned long long*>(a.early_logits) + static_cast<size_t>(row) * (a.early_stride / 2U);
    uint32_t key[PER];
    uint64_t missing = ~0ULL;
    for (uint32_t spins = 0; spins < kEarlySpinLimit && missing; ++spins) {
        bool mine = false;
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t e = lane + 64U * i;
            key[i] = 0;                                                          // 0 = absent or taken
            if (e < E) {
                const unsigned long long word = __hip_atomic_load(z + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);       // written by other workgroups of this launch
                mine = mine || static_cast<uint32_t>(word >> 32) != epoch;
                const uint32_t b = static_cast<uint32_t>(word);
                const uint32_t sortable = (b & 0x80000000U) ? ~b : (b | 0x80000000U);
                key[i] = sortable ? sortable : 1U;
            }
        }
        missing = __ballot(mine);
        if (missing) __builtin_amdgcn_s_sleep(4);
    }
    ok = missing == 0;
    uint32_t my_id = 0;
#pragma unroll 1
    for (uint32_t k = 0; k < K; ++k) {
        uint32_t best = key[0];
#pragma unroll
        for (uint32_t i = 1; i < PER; ++i) best = key[i] > best ? key[i] : best;
        best = max_wave_u32(best);
        uint32_t id = 0;
        bool found = false;
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const uint64_t holders = __ballot(key[i] == best);
            if (!found && holders) {
                found = true;
                const uint32_t owner = static_cast<uint32_t>(__ffsll(static_cast<long long>(holders))) - 1U;
                id = owner + 64U * i;
                if (lane == owner) key[i] = 0;
            }
        }
        if (lane == k) my_id = id;
    }
    return my_id;
}
__device__ __forceinline__ uint32_t early_select_row(const RouteArgs& a, uint32_t row, uint32_t epoch, bool& ok) {
    const uint32_t E = a.p.experts;
    if (E <= 128U) return early_select_row_per<2>(a, row, epoch, ok);
    if (E <= 256U) return early_select_row_per<4>(a, row, epoch, ok);
    if (E <= 512U) return early_select_row_per<8>(a, row, epoch, ok);
    return early_select_row_per<16>(a, row, epoch, ok);
}

// ---------------------------------------------------------------------------------------------------- the exact chain as a side block
// The reference's chain inside the layer launch: a one-wave block that owns two experts of one row. The two router-weight rows and the
// row itself come in chunks through the launch's two ring slots: chunks of 1024 features of fp16 / bf16 rows in two places (8 KB of weights and 2 KB of the
// row each), of 512 features of fp32 rows in three (4 KB and 2 KB). As many chunks as there are places are requested at the block's start - no row of
// hidden 2048 and 16 bits a value needs more -, and a place is filled anew when its chunk is through: the other waves of the launch saturate the memory, so
// what is awaited has to be asked for microseconds before. Lane 0 / 1 run the chains of the two experts, the weight operand by 128-bit LDS reads 48 features
// ahead; per 16 features one LDS read leaves feature k + t in lane t of every row of 16 lanes, widened once, and the fma takes it by a DPP row
// broadcast (chain_run of route_wave.hpp). (fp32 rows in registers before, all 128 of hidden 2048.)
// Needs hidden % 64 == 0.
constexpr uint32_t kSideExperts = 2, kSideSlotBytes = 10240;
template <int KIND> constexpr uint32_t side_chunk() { return KIND == 0 ? 512U : 1024U; }
template <int KIND> constexpr uint32_t side_places() { return KIND == 0 ? 3U : 2U; }

__device__ __forceinline__ void side_copy16(const void* src, uint32_t lds_at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_at), "v"(src) : "memory", "m0");
}

template <int KIND>
__device__ __forceinline__ void side_chain_block(lds_u8* ring0, lds_u8* ring1, const RouteArgs& a, uint32_t row, uint32_t e0) {
    constexpr uint32_t CHUNK = side_chunk<KIND>(), PLACES = side_places<KIND>(), SIZE = KIND == 0 ? 4U : 2U, WBYTES = 4U * CHUNK, XBYTES = SIZE * CHUNK;
    static_assert(XBYTES == 2048U && (PLACES == 2U ? 2U * WBYTES + XBYTES <= kSideSlotBytes : 4U * WBYTES + XBYTES <= kSideSlotBytes), "two ring slots hold the places");
    const uint32_t lane = threadIdx.x & 63U, chunks = (a.hidden + CHUNK - 1U) / CHUNK;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    // place p: weights of both experts, the row's values. Of the third one the weights lie behind the first, the values behind the second
    const auto weights_of = [&](uint32_t p) { return p == 1U ? ring1 : p == 0U ? ring0 : ring0 + 2U * WBYTES + XBYTES; };
    const auto values_of = [&](uint32_t p) { return p == 0U ? ring0 + 2U * WBYTES : p == 1U ? ring1 + 2U * WBYTES : ring1 + 2U * WBYTES + XBYTES; };
    const uint8_t* const xrow = a.x + row * a.x_stride;
    const float* wrow[kSideExperts];
#pragma unroll
    for (uint32_t i = 0; i < kSideExperts; ++i) wrow[i] = a.wr + static_cast<size_t>(e0 + i < a.p.experts ? e0 + i : a.p.experts - 1U) * a.hidden;
    // Every chunk is the same number of copies (the waits count them): pieces past the row's end fetch its last one again, into places that are never read.
    constexpr uint32_t WC = WBYTES / 1024U, XC = XBYTES / 1024U, COPIES = kSideExperts * WC + XC;
    const auto start = [&](uint32_t c, uint32_t p) {
        const uint32_t k0 = c * CHUNK, w_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(weights_of(p))), x_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(values_of(p)));
#pragma unroll
        for (uint32_t j = 0; j < WC; ++j) {
            const uint32_t k = k0 + 256U * j + 4U * lane, from = k < a.hidden ? k : a.hidden - 4U;
#pragma unroll
            for (uint32_t i = 0; i < kSideExperts; ++i) side_copy16(wrow[i] + from, w_at + WBYTES * i + 1024U * j);
        }
#pragma unroll
        for (uint32_t j = 0; j < XC; ++j) {
            const uint32_t k = k0 + 1024U / SIZE * j + 16U / SIZE * lane, from = k < a.hidden ? k : a.hidden - 16U / SIZE;
            side_copy16(xrow + static_cast<size_t>(SIZE) * from, x_at + 1024U * j);
        }
    };
    const auto widen = [&](uint32_t v) {
        if constexpr (KIND == 0) return f_of(v);
        else if constexpr (KIND == 1) return half_bits_to_float(v);
        else return f_of(v << 16);
    };
#pragma unroll
    for (uint32_t p = 0; p < PLACES; ++p)
        if (p < chunks) start(p, p);
    float acc = 0.0F;
    for (uint32_t c = 0, p = 0; c < chunks; ++c, p = p + 1U == PLACES ? 0U : p + 1U) {
        const uint32_t younger = chunks - 1U - c < PLACES - 1U ? chunks - 1U - c : PLACES - 1U;         // chunks asked for behind this one
        if (younger == 0U) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (younger == 1U) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(COPIES) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2U * COPIES) : "memory");
        const lds_u8* const w = weights_of(p) + (lane & 1U ? WBYTES : 0U);
        const lds_u8* const x = values_of(p) + SIZE * (lane & 15U);
        const uint32_t n = a.hidden - c * CHUNK < CHUNK ? a.hidden - c * CHUNK : CHUNK;
        // operands are fetched 48 features ahead of the chain (four buffers): with one step of 16 ahead every step waited for its
        // LDS reads (128 waits of ~200 cycles: the loop took 12.6 us inside the layer launch against ~5 us for the 2048 fmas).
        ChainStep S[4];
        uint32_t raw[4];         // the value of feature k + t as read; widened only when its 16 steps are about to run
        const auto load = [&](uint32_t s, uint32_t k) {
            typedef const __attribute__((address_space(3))) f32x4 lds_f32x4;
            typedef const __attribute__((address_space(3))) uint32_t lds_u32c;
            typedef const __attribute__((address_space(3))) uint16_t lds_u16c;
            const uint32_t kk = k < n ? k : n - 16U;            // (past the end: a valid place, never used)
#pragma unroll
            for (uint32_t i = 0; i < 4U; ++i) S[s].w[i] = *(lds_f32x4*)(w + 4U * kk + 16U * i);
            if constexpr (KIND == 0) raw[s] = *(lds_u32c*)(x + SIZE * kk);
            else raw[s] = *(lds_u16c*)(x + SIZE * kk);
        };
#pragma unroll
        for (uint32_t s = 0; s < 3U; ++s) load(s, 16U * s);
        for (uint32_t k = 0; k < n; k += 64U) {                 // hidden % 64 == 0 on this path
#pragma unroll
            for (uint32_t s = 0; s < 4U; ++s) {
                load((s + 3U) & 3U, k + 16U * (s + 3U));
                __builtin_amdgcn_sched_barrier(0);
                S[s].x = widen(raw[s]);
                acc = chain_run(S[s], acc);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (c + PLACES < chunks) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (every read of the place has returned)
            start(c + PLACES, p);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const uint32_t e = e0 + lane;
    if (lane < kSideExperts && e < a.p.experts)
        __hip_atomic_store(a.scores + static_cast<size_t>(row) * a.p.experts + e, a.bias ? acc + a.bias[e] : acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace strix950
