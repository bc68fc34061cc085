// Which kernel takes an FP8 projection of nine or more activation rows, and in
// which shape: rules over sizes only (fp8_batch.hip, fp8_gemv.hip).
#pragma once

#include <cstdint>

namespace plm {

constexpr int kPanelCols = 8;  // column tiles of 16 per workgroup of the panel kernel

// Activation rows from which the panel kernel is the faster one, for a launch of
// `outs` weights, the largest of `rows` rows, `blocks` blocks of 128 columns
// each.  The skinny kernel takes one launch, its time a step for each 16, 32 or
// 64 rows and for each round of workgroups; the panel kernel takes two to three
// launches (10 us and more) per weight but hardly grows.  Skinny / panel, us:
//   bf16   2048x7168 at 32, 33, 64 rows 20/21, 23/21, 33/23   2048x2048 at 64, 256 13/15, 16/24
//          7168x16384 at 64, 65 83/97, 121/97   4096x4096 at 64, 128, 192 21/26, 26/28, 48/43
//          24576x1536 at 64, 65 42/46, 62/46    7168x2048 at 64, 128, 192 17/30, 31/36, 45/31
//          2048 + 2048 x7168 at 64, 128, 192 34/41, 40/43, 77/67
//   fp32   2048x7168 at 16, 17 21/20, 24/20     2048x2048 at 64, 192, 256 12/14, 28/26, 28/27
//          7168x16384 at 32, 33 85/90, 122/90   4096x4096 at 32, 33, 65 21/24, 26/24, 38/35
//          24576x1536 at 32, 33 38/41, 56/42    7168x2048 at 64, 65 29/29, 36/27
//          2048 + 2048 x7168 at 64, 65, 96 40/39, 56/59, 76/60
//   2048 + 576 + 2048 x7168: bf16 at 64, 96, 128 40/58, 59/59, 76/60, fp32 at 33, 48, 64 41/53, 60/54, 74/55
//   4096 + 1024 + 1024 x4096: bf16 at 128, 192 50/57, 72/73, fp32 at 64, 96 47/48, 72/62
constexpr int64_t panel_from(int64_t rows, int64_t blocks, int outs, bool bf16) {
    if (outs > 1) {
        if (blocks < 32) return !bf16 && rows >= 2048 ? 193 : 257;
        return blocks >= 56 ? (bf16 ? 97 : 41) : (bf16 ? 193 : 65);
    }
    if (blocks < 32) {
        if (rows >= 16384) return bf16 ? 65 : 33;
        if (rows >= 4096 && blocks >= 16) return bf16 ? 129 : 65;
        return !bf16 && (rows >= 4096 || blocks >= 16) ? 193 : 257;
    }
    if (rows < 4096) return bf16 ? 33 : 17;
    return bf16 ? (blocks >= 56 ? 65 : 129) : 33;
}

// The same for the SwiGLU MLP.  Skinny / panel, us: bf16 7168/2048 at 64, 65
// 61/61, 78/61, 4096/1024 at 128, 129 35/39, 45/39, 1024/2048 at 256, 257 47/47,
// 56/42, 1024/512 at 512 25/32; fp32 7168/2048 at 32, 33 57/57, 64/58, 4096/1024
// at 64, 96 34/34, 39/37, 2048/1024 at 192, 256 39/41, 42/41, 7168/512 at 24, 32
// 39/37, 44/38: the skinny kernels' time grows with rows x weight (below 1024
// intermediate rows with rows x hidden), the panel's extra launches cost 10 to
// 15 us.
constexpr int64_t panel_mlp_from(int64_t hidden, int64_t inter, bool bf16) {
    if (!bf16 && hidden >= 7168 && inter < 1024) return 17;
    const int64_t size = hidden * (inter > 1024 ? inter : 1024);
    const int64_t rows = (int64_t(1) << (bf16 ? 29 : 28)) / size + 1, least = bf16 ? 65 : 33;
    return rows > least ? rows : least;
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
