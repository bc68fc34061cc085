// Which kernel takes an FP8 projection of nine or more activation rows, and in
// which shape: rules over sizes only (fp8_batch.hip, fp8_gemv.hip).
#pragma once

#include <cstdint>

namespace plm {

constexpr int kPanelCols = 8;  // column tiles of 16 per workgroup of the panel kernel

// Activation rows from which the panel kernel is the faster one, for a launch
// over `rows` weight rows.  The skinny kernel's time grows with the rows (us,
// bf16 / fp32 at 32, 64 and 128 rows: 7168x16384 53 / 80, 80 / 157, 155 / 310;
// 2048x7168 25 / 39, 38 / 39, 39 / 39), the panel kernel's hardly does
// (105 / 88, 23 / 23): they cross at about 80 / 36 rows of a tall weight and
// 32 / 14 of a short one, 68 / 36 for 24576x1536.
constexpr int64_t panel_from(int64_t rows, bool bf16) {
    return bf16 ? (rows >= 4096 ? 65 : 33) : (rows >= 4096 ? 33 : 17);
}

// Column tiles of m activation rows (two per token tile for hi and lo), in
// whole workgroups.
constexpr int panel_tiles(int64_t m, bool one_plane) {
    const int64_t tiles = (m + 15) / 16 * (one_plane ? 1 : 2);
    return static_cast<int>((tiles + kPanelCols - 1) / kPanelCols * kPanelCols);
}

// wr: 64 weight rows each a workgroup; splits: workgroups that share a tile's
// K slots (1: the slots stay together).
struct PanelPlan {
    int wr;
    int splits;
};

// Workgroups of 128 weight rows where that leaves one for each of the `cus`
// compute units, else of 64, and where those leave a quarter of the units idle
// the K slots split over two workgroups a unit: a workgroup alone takes 1.2 us a
// block whatever the launch, so 7168x16384 at 128 rows goes from 161 us (112
// workgroups) to 102, 2048x7168 from 77 to 24; 224 workgroups are better left
// whole (7168x16384 at 256 rows 167 us, split in three 214).
constexpr PanelPlan panel_plan(int64_t rows, bool silu, int64_t x_tiles, int waves, int cus) {
    const int64_t tile = silu ? 32 : 64, cols = x_tiles / kPanelCols;
    if ((rows + 2 * tile - 1) / (2 * tile) * cols >= cus) return {2, 1};
    const int64_t groups = (rows + tile - 1) / tile * cols;
    if (4 * groups >= 3 * static_cast<int64_t>(cus)) return {1, 1};
    const int64_t splits = (2 * cus + groups - 1) / groups;
    return {1, static_cast<int>(splits < waves ? splits : waves)};
}

}  // namespace plm
