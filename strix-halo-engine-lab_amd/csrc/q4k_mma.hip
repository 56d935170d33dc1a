// Experts on the int8 matrix cores (q4k_mma_moe.hpp): which instance serves a launch.
#include "host_common.hpp"
#include "launchers.hpp"
#include "q4k_mma_moe.hpp"

namespace strix950 {

// Tiles a workgroup runs over: as many as make about `most` stages, where a tile has few. The ring then starts once for all of them, but a
// workgroup's end is a step of the dispatch's balance, and the gate / up sweep (two matrices, 9 KB a stage) gains nothing from a longer
// run than eight stages. Measured (layer, run 1 | 2 | 4): hidden 2048 / ffn 768 / 128 experts top-8, 40 rows, project 117.9 | 121.3 | 127.2
// us, down (3 stages) 131.3 | 122.5 | 121.4; one rank's half of hidden 6144 / ffn 2560 / 160 experts, 16 rows, project 310.0 | 319.7 | 326.4,
// down (5 stages) 332.0 | 315.4 | 316.0; 1000 rows of the first (items of up to four sweeps), project 552.9 | 566.2 | 625.6, down 584.0 |
// 566.5 | 566.2.
inline uint32_t mma_run_tiles(uint32_t stages, uint32_t most, uint64_t tiles) {
    const uint32_t run = stages < most ? most / stages : 1U;
    const uint64_t full = tiles / (8ULL * compute_units());
    return run < full ? run : full > 1U ? static_cast<uint32_t>(full) : 1U;
}
struct MmaGrid { dim3 grid; MmaLaunch l; };
inline MmaGrid mma_grid(const mi355_moe_weights& w, uint32_t rows, uint32_t dense, uint32_t items, uint32_t tiles, uint32_t acts, uint32_t run) {
    return MmaGrid{dim3((tiles + run - 1U) / run, dense ? (dense + acts - 1U) / acts : items), MmaLaunch{rows * w.top_k, dense, tiles, run}};
}
// the rows of a dense batch at a stride of their own (every dense buffer and strided view; not the executor's pointer tables)
inline bool mma_direct(const A8Image& img, uint32_t dense) { return dense && img.per_row == 1U && !img.table; }
inline uint32_t mma_project_run(const mi355_moe_weights& w, uint32_t dense, uint32_t items) {
    return mma_run_tiles(w.hidden / 256U, 8U, static_cast<uint64_t>(w.ffn / 32U) * (dense ? 1U : items));
}
template <int FMT, int NAL, bool WIDE = false>
inline void launch_mma_project_nal(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, hipStream_t st) {
    const MmaGrid g = mma_grid(w, rows, dense, items, w.ffn / 32U, 2U * NAL, mma_project_run(w, dense, items));
    constexpr int DEPTH = NAL >= 8 ? 2 : 3, THREADS = 64 * mma_waves<2, WIDE>();
    if constexpr (FMT == kMmaQ4K && (WIDE || NAL < 16))
        if (mma_direct(r.in, dense)) { q4k_mma_project_kernel<FMT, NAL, DEPTH, true, WIDE><<<g.grid, THREADS, 0, st>>>(MmaArgs{w, r, g.l}); return; }
    q4k_mma_project_kernel<FMT, NAL, DEPTH, false, WIDE><<<g.grid, THREADS, 0, st>>>(MmaArgs{w, r, g.l});
}
// A launch with no more workgroups than compute units (few, long rows) runs four stages of a tile at a time (measured at 5120
// rows x 27648, 8 rows: 59 -> 33 us). Three slots a team where they hold up to eight rows and the matrix is long enough for the third to pay for its
// start: dense blocks over weights of more than 1 GB in turn, hidden | ffn, two, three slots, 4 and 8 rows: 4096 | 4096 27.7, 27.9 and 27.0, 27.5 us; 2048 |
// 8192 26.6, 26.5 and 27.8, 27.9; 6144 | 6144 35.2, 35.3 and 36.3, 36.3; 2048 | 16384 35.8, 34.9 and 40.5, 40.0; 8192 | 8192 43.3, 42.6 and 44.6, 44.1; 4096 |
// 14336 40.7, 40.0 and 47.8, 47.1; 5120 | 27648 73.7, 71.4 and 83.9, 80.9 (four slots 73.6 and 83.9). Sixteen rows are the same with two (102.3).
template <int FMT, int NAL>
inline void launch_mma_down_nal(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, hipStream_t st) {
    constexpr bool WIDE = mma_wide<FMT, NAL>();
    constexpr int THREADS = WIDE ? 512 : 256;
    const uint32_t tiles = w.hidden / (WIDE ? 2U * kMmaRows : kMmaRows);           // (the wide form: two at a time)
    const bool direct = mma_direct(r.h, dense);
    if constexpr (FMT == kMmaQ4K && !WIDE) {
        const MmaGrid g = mma_grid(w, rows, dense, items, tiles, 2U * NAL, 1U);
        if (static_cast<uint64_t>(g.grid.x) * g.grid.y <= compute_units()) {
            const auto launch = [&](auto slots) {
                constexpr int DEEP = decltype(slots)::value;
                if (direct) q4k_mma_down_kernel<FMT, NAL, DEEP, 4, true><<<g.grid, 1024, 0, st>>>(MmaArgs{w, r, g.l});
                else q4k_mma_down_kernel<FMT, NAL, DEEP, 4, false><<<g.grid, 1024, 0, st>>>(MmaArgs{w, r, g.l});
            };
            if (NAL <= 4 && static_cast<uint64_t>(tiles) * (w.ffn / 256U) >= 4096U) launch(std::integral_constant<int, NAL <= 4 ? 3 : 2>{});
            else launch(std::integral_constant<int, 2>{});
            return;
        }
    }
    const MmaGrid g = mma_grid(w, rows, dense, items, tiles, 2U * NAL, mma_run_tiles(w.ffn / 256U, NAL >= 8 ? 6U : 12U, static_cast<uint64_t>(tiles) * (dense ? 1U : items)));
    // (Q6_K: a fourth or sixth workgroup on a compute unit is worth more than a third slot: 24 rows of hidden 4096 / ffn 1536 / 64 experts
    // 178.3 -> 176.5 us; Q8_0, 40 rows of hidden 2048 / ffn 768 / 128 experts, 124.4 us with three slots, 126.5 with two)
    constexpr int DEPTH = NAL >= 8 || FMT == kMmaQ6K ? 2 : 3;
    if constexpr (FMT == kMmaQ4K)
        if (direct) { q4k_mma_down_kernel<FMT, NAL, DEPTH, 1, true><<<g.grid, THREADS, 0, st>>>(MmaArgs{w, r, g.l}); return; }
    q4k_mma_down_kernel<FMT, NAL, DEPTH, 1, false><<<g.grid, THREADS, 0, st>>>(MmaArgs{w, r, g.l});
}
// Gate / up rows past 16 activation rows: the wide form, or gate and up on one wavefront, which starts and ends a workgroup sooner (four wavefronts meet
// where eight do, and no register is spilled). So the line goes by the stages that a workgroup runs over, by rows an expert where they are few, and lies higher
// for Q5_K, whose wide form spills more. One wavefront against wide (time ratio; above one: wide is faster), rows an expert 18, 24, 32, 45, 64, 96:
//   Q4_K  160 experts of ffn 512    4 stages .89 .92 .97 1.01 1.03 1.11   6 .97 .99 1.03 1.04 1.07 1.10   8 1.00 1.02 1.06 1.08 1.07 1.12
//         80 experts of ffn 1536    4, runs of two tiles, 1.05 1.06 1.07 1.12 1.10 1.12   6 .96 .98 1.01 1.05 1.07 1.08   10 1.05 1.01 1.07 1.10 1.10 1.13
//         32 experts of ffn 1024    4 .96 .91 .95 1.02 1.05 1.06   6 .97 .99 1.03 1.05 1.07 1.06   8 .95 .97 1.05 1.05 1.06 1.11   16 1.10 1.09 1.14 1.12 1.14 1.16
//   Q5_K  160 experts of ffn 512    4 .83 .86 .90 .92 .97 1.06   6 .89 .93 .97 .96 .97 .98   8 .91 .95 .97 .99 .98 1.00   10 .96 .96 1.02 .99 1.03 1.05
//         80 experts of ffn 1536    4, runs of two tiles, .99 .97 1.00 .99 1.03 1.05   6 .90 .91 .94 .98 .96 .98   8 .91 .95 .93 .98 .98 1.03
//         32 experts of ffn 1024    4 .89 .89 .90 .97 .99 1.01   6 .93 .91 .97 1.02 1.03 1.07   8 .99 .96 1.04 1.06 1.09 1.11   12 1.06 1.08 1.15 1.14 1.13 1.14
// (95 experts top-6 of 1536 x 1536, Q5_K, 31 rows an expert: 231 us, wide 243; 128 experts of 2048 x 768, Q4_K, 62 rows: 327, wide 297.) Dense blocks are wide: 34
// and 48 rows, ffn 4096 1.11 1.10 (4 stages), 1.14 1.14 (7); 8192 .99 .98, 1.01 .99; 16384 .98 1.02, 1.04 1.08; 28672 1.00 1.04, 1.05 1.08.
template <int FMT>
inline bool mma_project_wide(const mi355_moe_weights& w, uint32_t rows, uint32_t dense, uint32_t run) {
    const uint32_t stages = w.hidden / 256U;
    if (dense) return true;
    const uint64_t steps = static_cast<uint64_t>(stages) * run, rows_of_all = static_cast<uint64_t>(rows) * w.top_k;
    if (FMT == kMmaQ5K) return stages >= 12U || steps * rows_of_all >= 400ULL * w.experts;
    return steps >= 8U || steps * rows_of_all >= 180ULL * w.experts;
}
template <int FMT>
inline void launch_mma_project_format(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, uint32_t width, hipStream_t st) {
    if (width <= 4U) launch_mma_project_nal<FMT, 2>(w, r, rows, dense, items, st);
    else if (width <= 8U) launch_mma_project_nal<FMT, 4>(w, r, rows, dense, items, st);
    else if (width <= 16U) launch_mma_project_nal<FMT, 8>(w, r, rows, dense, items, st);
    else if (mma_project_wide<FMT>(w, rows, dense, mma_project_run(w, dense, items))) launch_mma_project_nal<FMT, 16, true>(w, r, rows, dense, items, st);
    else launch_mma_project_nal<FMT, 16>(w, r, rows, dense, items, st);
}
// (rows of another format: sixteen activation rows to a sweep at most, whose two halves of a group take the result registers of 32)
template <int FMT>
inline void launch_mma_down_format(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, uint32_t width, hipStream_t st) {
    if (width <= 4U) launch_mma_down_nal<FMT, 2>(w, r, rows, dense, items, st);
    else if (width <= 8U) launch_mma_down_nal<FMT, 4>(w, r, rows, dense, items, st);
    else {
        // The wide form from a workgroup per compute unit on: dense 8192 x 4096, 64 rows (256 workgroups) 25.8 -> 23.7 us; with fewer its stages, of
        // twice the rows, follow one another in fewer places (5120 x 27648, 32 | 64 rows, 80 | 160 workgroups 81 | 109 us against 115 | 116).
        const uint64_t groups = static_cast<uint64_t>(w.hidden / (2U * kMmaRows)) * (dense ? (dense + 31U) / 32U : items);
        if constexpr (mma_wide<FMT, 16>())
            if (width > 16U && groups >= compute_units()) return launch_mma_down_nal<FMT, 16>(w, r, rows, dense, items, st);
        launch_mma_down_nal<FMT, 8>(w, r, rows, dense, items, st);
    }
}
// width: the most rows an item (or the dense batch) holds
void launch_mma_project(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, uint32_t width, hipStream_t st) {
    if (w.gate_type == MI355_TYPE_Q5_K) launch_mma_project_format<kMmaQ5K>(w, r, rows, dense, items, width, st);
    else launch_mma_project_format<kMmaQ4K>(w, r, rows, dense, items, width, st);
}
void launch_mma_down(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, uint32_t dense, uint32_t items, uint32_t width, hipStream_t st) {
    if (w.down_type == MI355_TYPE_Q6_K) launch_mma_down_format<kMmaQ6K>(w, r, rows, dense, items, width, st);
    else if (w.down_type == MI355_TYPE_Q8_0) launch_mma_down_format<kMmaQ80>(w, r, rows, dense, items, width, st);
    else if (w.down_type == MI355_TYPE_Q5_1) launch_mma_down_format<kMmaQ51>(w, r, rows, dense, items, width, st);
    else launch_mma_down_format<kMmaQ4K>(w, r, rows, dense, items, width, st);
}
void launch_mma_gate_up_rows(const mi355_moe_weights& w, const RowsK& r, uint32_t rows, hipStream_t st) {
    const uint32_t tiles = w.ffn / kMmaRows;
    const MmaLaunch l{rows * w.top_k, rows, tiles, 1U};
    const dim3 grid(tiles, 1, 2);
    const auto launch = [&](auto direct) {
        constexpr bool D = decltype(direct)::value;
        if (rows <= 8U) q4k_mma_down_kernel<kMmaQ4K, 4, 3, 1, D, true><<<grid, 256, 0, st>>>(MmaArgs{w, r, l});
        else q4k_mma_down_kernel<kMmaQ4K, 8, 2, 1, D, true><<<grid, 256, 0, st>>>(MmaArgs{w, r, l});
    };
    if (mma_direct(r.in, rows)) launch(std::true_type{});
    else launch(std::false_type{});
}

}  // namespace strix950
