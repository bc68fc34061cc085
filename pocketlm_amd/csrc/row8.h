// row8-packed GEMV launcher shared by the kernels of row8.hip and the dense
// decode layer of kv_cache.hip.
#pragma once

#include "common.h"

namespace plm {

// One matrix of a fused row8 launch: packed[blk][k][lane] = W[8*blk + lane][k].
struct Row8Mat {
    const uint16_t* packed;
    const uint16_t* bias;  // may be null
    float* out;
    int64_t rows;
    int64_t first_tile = 0;    // filled in by row8_gemv
    // Epilogue: when out16 is set, out16[row] = storage(resid[row] + y[row])
    // (rounded as the reference's write_u16) and `out` is not written.
    const float* resid = nullptr;
    uint16_t* out16 = nullptr;
};

// The activation vector of a row8 launch (one of):
//   u16            fp16/bf16 values;
//   u16 + norm_w   storage(u16 * (1 / sqrt(mean(u16^2) + eps)) * norm_w), the
//                  reference's rms_norm_one rounded to the storage type;
//   f32            fp32 values;
//   f32 + f32_b    f32 / (1 + exp(-f32)) * f32_b (SiLU(gate) * up).
struct Row8X {
    const uint16_t* u16 = nullptr;
    const uint16_t* norm_w = nullptr;
    float eps = 0.0f;
    const float* f32 = nullptr;
    const float* f32_b = nullptr;
};

constexpr int kRow8MaxMats = 8;

// out_i = W_i x (+ bias_i) for up to kRow8MaxMats matrices sharing x, in one
// launch on `st`.  x is fp16/bf16 (hidden) or fp32 (hidden_f32, hidden null).
int row8_gemv(const uint16_t* hidden, const float* hidden_f32, const Row8Mat* mats, int n, int64_t K, int dtype_code,
              hipStream_t st);
int row8_gemv_x(const Row8X& x, const Row8Mat* mats, int n, int64_t K, int dtype_code, hipStream_t st);

// Waves of a GEMV workgroup over K columns: min(K / 64 rounded up, kRow8Waves).
constexpr int kRow8Waves = 8;

// ------------------------------------------------------------------ many rows (row8_batch.hip)
//
// Up to kRow8BatchRows activation rows against row8 weights on the matrix
// cores.  The activations come as planes of storage-type values whose sum is
// the row (one plane for fp16 / bf16 rows; fp32 rows as kRow8Parts parts),
// in the order the lanes of the kernel read them: 16-byte pieces
// [K / 32][token tile][q = 0..3][token of the tile], piece (g, q) of a row
// being its columns 32 g + 4 j + q, j = 0..7 (one load of a lane's weights
// holds one column of its 8 rows).
constexpr int kRow8BatchRows = 128;
constexpr int kRow8Parts = 3;
// 16-row token tiles of an activation plane (rows past m may hold anything).
constexpr int row8_token_tiles(int64_t m) { return m <= 16 ? 1 : (m <= 32 ? 2 : (m <= 64 ? 4 : 8)); }
constexpr int64_t row8_plane_bytes(int64_t m, int64_t K) { return K / 32 * row8_token_tiles(m) * 1024; }

struct Row8BatchMat {
    const uint16_t* packed;
    int64_t rows;      // a multiple of 8
    int64_t out_col;   // first column of the output
    int64_t first_tile = 0;
};

// part[s][m][out_col + row] = sum over K slice s of x_m W[row], times
// inv[m] when inv is set.
struct Row8Batch {
    Row8BatchMat mats[3];
    int nmats = 0;
    const uint16_t* x = nullptr;   // planes, row8_plane_bytes each
    const float* inv = nullptr;
    float* part = nullptr;         // [splits][m][ld]
    int64_t ld = 0;                // a multiple of 4
    int64_t K = 0;                 // a multiple of 32
    int planes = 1;
    int m = 0;                     // at most kRow8BatchRows
    int splits = 1;                // of row8_batch_splits
    int dtype_code = 0;
};

// K slices of a launch over `rows` weight rows in all.
int row8_batch_splits(int64_t rows, int64_t K);
int row8_batch(const Row8Batch& p, hipStream_t st);

}  // namespace plm
