// The expert plan (plan_layout.hpp): a workgroup per expert, as a launch of its own or in front of the workgroups that prepare a batch's rows.
//
// Every workgroup counts all assignments by expert (LDS), so it knows by itself where its expert's assignments and work items begin, and places
// its own assignments: a wavefront owns a contiguous share of them, ballots give each one's rank. Bound by latency (two reads of the
// routes). Measured as part of the launch that prepares the rows, against a workgroup that planned alone, a launch that ordered and that launch
// without the plan: 333 rows top-8 over 128 experts (prefill) 4.9 us against 4.8 + 4.8 + 4.9, 1000 rows over 256 8.2 against 6.4 + 7.2 + 5.4, 4000
// rows over 128 18.6 against 14.9 + 22.1 + 6.2. (One workgroup that ordered as well, in front of the rows' ones: 7.3, 14.5, 37.)
#pragma once
#include "device_math.hpp"
#include "plan_layout.hpp"
#include "route_wave.hpp"

namespace strix950 {

// The routes of a batch as the plan kernels read them: assignment a = row a / top_k, slot a % top_k, rows `rs` bytes apart.
struct RoutesView {
    const uint32_t* base;
    uint64_t rs;
    uint32_t top_k;
    __device__ __forceinline__ const uint32_t* place(uint32_t a) const {
        if (rs == 4ULL * top_k) return base + a;
        const uint32_t row = a / top_k;
        return reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(base) + row * rs) + (a - row * top_k);
    }
    __device__ __forceinline__ uint32_t at(uint32_t a) const { return *place(a); }
};
inline RoutesView dense_routes(const uint32_t* routes, uint32_t top_k) { return RoutesView{routes, 4ULL * top_k, top_k}; }

struct PlanArgs { RoutesView routes; uint32_t experts, assignments, split, item_bound; uint32_t* plan; };      // (no experts: no plan, nothing else is read)

// Inclusive prefix sum over a wavefront: row shifts inside the rows of 16, then the rows' totals by row broadcasts (DPP, no LDS).
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x111, 0xF, 0xF, false));      // row_shr:1
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x112, 0xF, 0xF, false));      // row_shr:2
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x114, 0xF, 0xF, false));      // row_shr:4
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x118, 0xF, 0xF, false));      // row_shr:8
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x142, 0xA, 0xF, false));      // row_bcast:15 into rows 1 and 3
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x143, 0xC, 0xF, false));      // row_bcast:31 into rows 2 and 3
    return v;
}

// What workgroup e shares: the counts of all experts, and per wavefront the sums over the experts below e (assignments, items, touched experts) and
// this expert's assignments; workgroup 0: the sums over all of them as well.
struct PlanLds {
    uint32_t count[kRouteMaxExperts];
    u32x4 below[16], all[16];
    uint32_t mine[16];
};

// Expert e's part of the plan, by a workgroup of any whole number of wavefronts up to 16.
__device__ __forceinline__ void plan_block(PlanLds& lds, const PlanArgs& p, uint32_t e) {
    const uint32_t tid = threadIdx.x, threads = blockDim.x, lane = tid & 63U, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = threads >> 6;
    const uint32_t experts = p.experts, assignments = p.assignments;
    for (uint32_t i = tid; i < experts; i += threads) lds.count[i] = 0;
    const uint32_t share = ((assignments + waves - 1U) / waves + 63U) & ~63U;
    const uint32_t lo = wave * share < assignments ? wave * share : assignments, hi = assignments - lo < share ? assignments : lo + share;
    // turn(key, a): the wavefront's assignments in order, 64 at a time (key = experts: none, or of no expert); eight turns asked for together
    const auto walk = [&](auto turn) __attribute__((always_inline)) {
        constexpr uint32_t TURNS = 8;
#pragma unroll 1
        for (uint32_t a0 = lo; a0 < hi; a0 += 64U * TURNS) {
            uint32_t key[TURNS];
#pragma unroll
            for (uint32_t t = 0; t < TURNS; ++t) {
                const uint32_t a = a0 + 64U * t + lane;
                key[t] = a < hi ? p.routes.at(a) : experts;
            }
#pragma unroll
            for (uint32_t t = 0; t < TURNS; ++t) turn(key[t], a0 + 64U * t + lane);
        }
    };
    uint32_t mine = 0;
    __syncthreads();
    walk([&](uint32_t key, uint32_t) {
        if (key < experts) atomicAdd(&lds.count[key], 1U);
        mine += static_cast<uint32_t>(__popcll(__ballot(key == e)));
    });
    __syncthreads();
    uint32_t sums[3] = {0U, 0U, 0U}, totals[3] = {0U, 0U, 0U}, most = 0;
    for (uint32_t i = tid; i < experts; i += threads) {
        const uint32_t c = lds.count[i], v[3] = {c, (c + p.split - 1U) / p.split, c != 0 ? 1U : 0U};
#pragma unroll
        for (int k = 0; k < 3; ++k) { sums[k] += i < e ? v[k] : 0U; totals[k] += v[k]; }
        most = c > most ? c : most;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) sums[k] = wave_inclusive_scan(sums[k]);
    if (lane == 63U) { lds.below[wave] = u32x4{sums[0], sums[1], sums[2], 0U}; lds.mine[wave] = mine; }
    if (e == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) totals[k] = wave_inclusive_scan(totals[k]);
#pragma unroll
        for (int d = 32; d; d >>= 1) {
            const uint32_t other = __shfl_xor(most, d);
            most = other > most ? other : most;
        }
        if (lane == 63U) lds.all[wave] = u32x4{totals[0], totals[1], totals[2], most};
    }
    __syncthreads();
    uint32_t first = 0, item = 0, touched = 0, before = 0;
    for (uint32_t w = 0; w < waves; ++w) {
        const u32x4 t = lds.below[w];
        first += t.x; item += t.y; touched += t.z;
        before += w < wave ? lds.mine[w] : 0U;
    }
    const uint32_t c = lds.count[e], pieces = (c + p.split - 1U) / p.split;
    uint32_t* const items = p.plan + plan_items_at(experts, assignments);
    for (uint32_t i = tid; i < pieces; i += threads) {
        const uint32_t b = i * p.split;
        *reinterpret_cast<uint4*>(items + 4U * (item + i)) = make_uint4(e, first + b, first + (b + p.split < c ? b + p.split : c), 0U);
    }
    if (tid == 0) {
        p.plan[kPlanOffsetsAt + e] = first;
        if (c != 0) p.plan[plan_touched_at(experts) + touched] = e;
    }
    if (e == 0) {
        u32x4 all = {0U, 0U, 0U, 0U};
        for (uint32_t w = 0; w < waves; ++w) {
            const u32x4 t = lds.all[w];
            all.x += t.x; all.y += t.y; all.z += t.z; all.w = t.w > all.w ? t.w : all.w;
        }
        for (uint32_t u = all.y + tid; u < p.item_bound; u += threads) *reinterpret_cast<uint4*>(items + 4U * u) = make_uint4(0U, 0U, 0U, 0U);
        if (tid == 0) {
            p.plan[kPlanOffsetsAt + experts] = all.x;
            p.plan[0] = assignments; p.plan[1] = all.z; p.plan[2] = all.w; p.plan[4] = all.y;
        }
    }
    uint32_t* const order = p.plan + plan_order_at(experts);
    uint32_t at = first + before;
    if (mine != 0)
        walk([&](uint32_t key, uint32_t a) {
            const uint64_t votes = __ballot(key == e);
            if (key == e) order[at + static_cast<uint32_t>(__popcll(votes & ((1ULL << lane) - 1ULL)))] = a;
            at += static_cast<uint32_t>(__popcll(votes));
        });
}

}  // namespace strix950
