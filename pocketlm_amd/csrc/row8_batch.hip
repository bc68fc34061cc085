// Many activation rows against row8-packed fp16/bf16 weights on the matrix
// cores (gfx950): the projections of a prompt through a dense layer.
//
// row8 stores the 8 rows of a block side by side at each column, the
// transpose of what an MFMA operand wants (8 columns of one row per lane).
// So lane l holds a whole 8-row block: block l & 15 of the wave's 16 (128
// weight rows), columns 4 j + (l >> 4) of a 32-column step in load j (64
// contiguous bytes per block and load), and after 32 register permutes its
// eight operands are rows t = 0..7 of that block: MFMA t takes row t of all
// 16 blocks.  No LDS; the activations are stored in the order the lanes read
// them (row-major activation planes, 64-byte pieces of 16 rows a load, were
// the bound: gate + up 135 us and down 139 against 112 and 99).
//
// A workgroup's KS x TG waves: TG groups of token tiles share the weights
// through the caches, KS parts of the K slice meet in LDS.
//
// The sums are as close to 64 bits as the one-row GEMV's (row8.hip).  A matrix
// instruction adds its 32 products to C in several roundings, and cuts off
// what of C, or of the products, lies below the largest of them, always
// downwards: a running sum in C is 2.7e-7 off over 3584 columns and the small
// parts of fp32 activations under the large ones 2.2e-7 over 18944.  So each
// 32-column step starts from zero, the small parts have a result of their own,
// and vector instructions add the results; slices keep a wave's chain of adds
// short.  RMS error over RMS value here / one-row GEMV, 120 rows:
//   fp16  q k v 4608x3584 8.9e-8 / 9.8e-8   gate up 37888x3584 9.7e-8 / 9.6e-8
//         o 3584x3584 1.01e-7 / 1.00e-7     down 3584x18944 1.44e-7 / 1.40e-7
//   bf16  8.1e-8 / 8.3e-8, 9.1e-8 / 8.2e-8, 9.7e-8 / 1.00e-7, 1.35e-7 / 1.42e-7
//
// What bounds it: loads in flight and their spread.  At 120 rows of a 3584 /
// 18944 layer in fp16 (us): q + k + v 27, o 29, gate + up 126 (2.2 TB/s),
// down 113.  Sums kept in the matrix instruction and two fp16 parts took 27,
// 25, 112 and 94.  The whole layer 13.6 ms one row at a time -> 0.39 ms of
// kernels.
#include <algorithm>
#include <cstring>

#include "fp8_mfma.h"
#include "row8.h"

namespace {

using plm_fp8::plm_f32x4;
using plm_fp8::run_pipelined;
typedef _Float16 plm_f16x8 __attribute__((ext_vector_type(8)));

constexpr int kTileRows = 128;

struct Row8BatchArgs {
    plm::Row8BatchMat mats[3];
    const uint16_t* x;
    const float* inv;
    float* part;
    int64_t ld;
    int64_t K;
    int nmats;
    int m;
    int tiles;   // row tiles of all matrices
    int splits;
};

template <bool BF16>
__device__ __forceinline__ plm_f32x4 mfma16(plm_u32x4 a, plm_u32x4 b, plm_f32x4 c) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(plm_fp8::plm_bf16x8, a),
                                                       __builtin_bit_cast(plm_fp8::plm_bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(plm_f16x8, a),
                                                      __builtin_bit_cast(plm_f16x8, b), c, 0, 0, 0);
}

template <bool BF16, int TB, int PL, int KS, int P, int TG>
__global__ __launch_bounds__(64 * KS * TG, TG > 1 ? 2 : 1) void row8_batch_kernel(const Row8BatchArgs a) {
    constexpr int RB = TB * TG < 4 ? TB : (TG >= 4 ? 1 : 4 / TG);  // token tiles per round of the waves' sums
    __shared__ plm_f32x4 sums[TG * (KS > 1 ? KS / 2 : 1) * 8 * RB * 64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tg = wave % TG, ks = wave / TG;
    const int lane = threadIdx.x & 63;
    const int li = lane & 15, qd = lane >> 4;
    const int split = blockIdx.x % a.splits, tile = blockIdx.x / a.splits;
    int mi = 0;
    for (int i = 1; i < a.nmats; ++i)
        if (tile >= a.mats[i].first_tile) mi = i;
    const plm::Row8BatchMat mat = a.mats[mi];
    const int64_t blk0 = (tile - mat.first_tile) * (kTileRows / 8);
    const int64_t blocks = mat.rows / 8;
    // blocks past the end read the last one; their results are dropped
    const char* wp = reinterpret_cast<const char*>(mat.packed) + (min(blk0 + li, blocks - 1) * a.K + qd) * 16;
    // the lane's 16 bytes of a step's first token tile; tiles are 1 KB apart
    const char* xp = reinterpret_cast<const char*>(a.x) + tg * TB * 1024 + lane * 16;
    const int64_t plane = a.K / 32 * TB * TG * 1024;
    // this wave's 32-column steps: part ks of slice `split` of the row
    const int64_t steps = a.K / 32;
    const int64_t parts = static_cast<int64_t>(a.splits) * KS, part = static_cast<int64_t>(split) * KS + ks;
    const int64_t s0 = steps * part / parts;
    const int nk = static_cast<int>(steps * (part + 1) / parts - s0);
    // tiles start at different steps, so that they do not walk the columns (and
    // with them the memory channels) in step: down 3584x18944 110 -> 99 us
    const int rot = (tile * 5) % max(nk, 1);

    plm_f32x4 acc[8][TB];
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) acc[t][tb] = plm_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    plm_u32x4 q[P][8], x[P][PL][TB];
    auto issue = [&](int slot, int k) {
        int kk = k + rot;
        kk = kk >= nk ? kk - nk : kk;
        const int64_t s = s0 + kk;
#pragma unroll
        for (int j = 0; j < 8; ++j) q[slot][j] = plm_fp8::xload16(wp + s * 512 + 64 * j);
#pragma unroll
        for (int pl = 0; pl < PL; ++pl)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) x[slot][pl][tb] = plm_fp8::xload16(xp + pl * plane + (s * TB * TG + tb) * 1024);
    };
    auto compute = [&](int slot, int) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            // row t of the block: its value of column j in load j
            plm_u32x4 w;
#pragma unroll
            for (int d = 0; d < 4; ++d)
                w[d] = __builtin_amdgcn_perm(q[slot][2 * d + 1][t >> 1], q[slot][2 * d][t >> 1],
                                             (t & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
                const plm_f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
                plm_f32x4 d = mfma16<BF16>(w, x[slot][0][tb], none);
                if constexpr (PL > 1) {
                    plm_f32x4 small = none;
#pragma unroll
                    for (int pl = PL - 1; pl >= 1; --pl) small = mfma16<BF16>(w, x[slot][pl][tb], small);
                    d = d + small;
                }
                acc[t][tb] = acc[t][tb] + d;
            }
        }
    };
    run_pipelined<P>(nk, issue, compute);

#pragma unroll
    for (int half = KS / 2; half >= 1; half /= 2) {
#pragma unroll
        for (int r = 0; r < TB; r += RB) {
            if (ks >= half && ks < 2 * half) {
#pragma unroll
                for (int t = 0; t < 8; ++t)
#pragma unroll
                    for (int tb = 0; tb < RB; ++tb)
                        sums[(((tg * half + ks - half) * 8 + t) * RB + tb) * 64 + lane] = acc[t][r + tb];
            }
            __syncthreads();
            if (ks < half) {
#pragma unroll
                for (int t = 0; t < 8; ++t)
#pragma unroll
                    for (int tb = 0; tb < RB; ++tb)
                        acc[t][r + tb] = acc[t][r + tb] + sums[(((tg * half + ks) * 8 + t) * RB + tb) * 64 + lane];
            }
            __syncthreads();
        }
    }
    if (ks != 0) return;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const int m = 16 * (tg * TB + tb) + li;
        if (m >= a.m) continue;
        const float f = a.inv != nullptr ? a.inv[m] : 1.0f;
        float* o = a.part + (static_cast<int64_t>(split) * a.m + m) * a.ld + mat.out_col;
        // D: lane (token li, blocks 4 qd + j), row t of the block
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t blk = blk0 + 4 * qd + j;
            if (blk >= blocks) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                plm_f32x4 v;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = acc[4 * h + i][tb][j] * f;
                *reinterpret_cast<plm_f32x4*>(o + blk * 8 + 4 * h) = v;
            }
        }
    }
}

template <bool BF16, int TB, int PL, int KS, int P, int TG = 1>
int launch(const Row8BatchArgs& a, hipStream_t st) {
    hipLaunchKernelGGL((row8_batch_kernel<BF16, TB, PL, KS, P, TG>), dim3(static_cast<unsigned>(a.tiles * a.splits)),
                       dim3(64 * KS * TG), 0, st, a);
    return plm::check_launch("row8 batch kernel");
}

// Steps in flight (P), waves that split a slice (KS) and token groups (TG) by
// token tiles.  A wave holds at most 4 token tiles (128 accumulators): the
// adds need them in vector registers, and two waves share a SIMD (q + k + v
// 30 -> 27 us against one wave with 8 tiles).  Several planes: groups of 2
// tiles; three steps of three planes in flight do not fit the registers.
template <bool BF16, int PL>
int launch_m(const Row8BatchArgs& a, hipStream_t st) {
    const int tiles = plm::row8_token_tiles(a.m);
    if (tiles == 1) return launch<BF16, 1, PL, 4, 3>(a, st);
    if (tiles == 2) return launch<BF16, 2, PL, 4, 3>(a, st);
    if constexpr (PL == 1) {
        if (tiles == 4) return launch<BF16, 4, PL, 2, 2>(a, st);
        return launch<BF16, 4, PL, 2, 2, 2>(a, st);
    } else {
        if (tiles == 4) return launch<BF16, 2, PL, 2, 2, 2>(a, st);
        return launch<BF16, 2, PL, 1, 2, 4>(a, st);
    }
}

}  // namespace

// A power of two up to 16 (so that the workgroups of one slice, which share
// its activations, land on the same XCDs): as many as keep two workgroups per
// compute unit and 8 steps per slice, and for the sums' error as many as keep a
// slice to 16 steps up to four slices, to 32 beyond (gate + up 37888x3584 in
// one slice 1.5e-7 off 64 bits, in four 9.7e-8).
int plm::row8_batch_splits(int64_t rows, int64_t K) {
    const int64_t tiles = std::max<int64_t>(1, plm::ceil_div(rows, kTileRows)), steps = K / 32;
    auto more = [&](int s) {
        return (2 * s * tiles <= 2 * plm::cu_count() && steps >= 2 * s * 8) || steps > (s < 4 ? 16 : 32) * s;
    };
    int s = 1;
    while (s < 16 && more(s)) s *= 2;
    return s;
}

int plm::row8_batch(const Row8Batch& p, hipStream_t st) {
    Row8BatchArgs a;
    std::memset(&a, 0, sizeof(a));
    if (p.m < 1 || p.m > kRow8BatchRows || p.K % 32 != 0 || p.ld % 4 != 0 || p.splits < 1)
        return plm::fail(2, "row8 batch: bad dimensions");
    int64_t tiles = 0;
    for (int i = 0; i < p.nmats; ++i) {
        if (!plm::aligned16(p.mats[i].packed)) return plm::fail(2, "packed weight not 16-byte aligned");
        if (p.mats[i].rows < 8 || p.mats[i].rows % 8 != 0 || p.mats[i].out_col % 4 != 0)
            return plm::fail(2, "row8 batch: bad dimensions");
        a.mats[i] = p.mats[i];
        a.mats[i].first_tile = tiles;
        tiles += plm::ceil_div(p.mats[i].rows, kTileRows);
    }
    a.nmats = p.nmats;
    a.x = p.x;
    a.inv = p.inv;
    a.part = p.part;
    a.ld = p.ld;
    a.K = p.K;
    a.m = p.m;
    a.tiles = static_cast<int>(tiles);
    a.splits = p.splits;
    if (tiles * p.splits > 0x7FFFFFFF) return plm::fail(2, "too many row tiles");
    if (p.dtype_code == 1) {
        if (p.planes == 1) return launch_m<true, 1>(a, st);
        if (p.planes == kRow8Parts) return launch_m<true, kRow8Parts>(a, st);
    } else {
        if (p.planes == 1) return launch_m<false, 1>(a, st);
        if (p.planes == kRow8Parts) return launch_m<false, kRow8Parts>(a, st);
    }
    return plm::fail(2, "row8 batch: bad plane count");
}
