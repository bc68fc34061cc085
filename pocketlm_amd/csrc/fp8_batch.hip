// FP8 block-scaled projections of nine or more activation rows on gfx950:
// a prompt chunk through linear / dual / SwiGLU weights, and the (expert,
// row) pairs of a prompt chunk through the routed experts.
//
// fp8_batch_kernel reads each weight byte once for up to 16 TB activation
// rows, where the kernels of fp8_gemv.hip take 8 rows per pass.  Tiles are
// whole MFMA tiles: A = 16 weight rows, B = 16 activation rows, one half (64
// columns) of a 128-column block per MFMA pair.  Lane l holds the 16 weight
// bytes at columns 64 h + 16 (l >> 4) of weight row l & 15 and the same
// columns of activation row l & 15, so the products of a (weight row,
// activation row, half) meet in the same MFMA positions as in fp8_gemv.hip,
// where the two halves sit in rows of their own.  The blocks are dealt to the
// waves alike, each block's D is scaled into the half's accumulator, halves
// and then waves are added in the same order: a row's result has the bits of
// a one-row call.
//
// Measured on an MI355X against passes of 8 rows: 7168x16384 at 16 bf16 rows
// 61 -> 45 us, at 64 rows 212 -> 83 us, 2048x7168 at 9 and 16 rows 14.4 -> 11.4
// and 16.1 -> 13.6; 96 rows of top-8 over 256 experts of 7168/2048 27.2 -> 2.02
// ms (5.3 TB/s: the weights of every chosen expert, read once).
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "fp8_batch.h"
#include "fp8_mfma.h"

namespace {

using namespace plm_fp8;

enum XKind { kXF32 = 0, kXBf16 = 1, kXPlanes = 2 };

struct BatchArgs {
    const uint8_t* w[2][plm::kBatchGroups];
    const float* s[2][plm::kBatchGroups];
    const char* x;
    const char* xlo;
    int64_t x_stride;  // bytes
    float* out;
    uint16_t* hhi;
    uint16_t* hlo;
    int64_t rows;
    int64_t K;
    int64_t scale_cols;
    int64_t m;
    int64_t list_ld;
    const int* count;
    const int* base;
    const int* list;
    int tiles;    // row tiles per group
    int nblocks;  // 128-column blocks per row
    int tiled;
    int nouts;    // groups with rows and outputs of their own
    int64_t out_rows[plm::kBatchOuts];
    float* outs[plm::kBatchOuts];
};

// A workgroup owns 16 TA rows of each of its NWT weights; wave w of nw takes
// the K blocks w, w + nw, ... for all 16 TB activation rows of a pass.
template <int TA, int TB, int P, int NWT, bool SILU, int XM, int MAXW>
__global__ __launch_bounds__(64 * MAXW) void fp8_batch_kernel(const BatchArgs a) {
    constexpr int NT = NWT * TA;
    constexpr int PL = XM == kXPlanes ? 2 : 1;  // planes of the activations, with accumulators of their own
    constexpr bool XB = XM != kXF32;
    constexpr int XE = XB ? 2 : 4;
    // Whether a ragged block's columns past K are masked before its first
    // matrix instruction, and not half by half: with the branch between one and
    // the read of its result ROCm 7.2's compiler left out the wait states in a
    // 16-row instance (wrong sums after a NaN byte); in the wider ones it does
    // not, and there the early mask is slower (the 4096/2048 MLP at 17 rows 24
    // -> 32 us).
    constexpr bool EARLY = TA == 1 && !SILU;
    extern __shared__ plm_f32x4 red[];  // [wave][tile][lane]
    const int nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int li = lane & 15, qd = lane >> 4;
    const int g = blockIdx.x / a.tiles;
    const int64_t row0 = static_cast<int64_t>(blockIdx.x - g * a.tiles) * 16 * TA;
    const int64_t count = a.count != nullptr ? a.count[g] : a.m;
    int64_t obase = a.base != nullptr ? a.base[g] : g * a.m;
    int64_t rows = a.rows;
    float* out = a.out;
    if (!SILU && XM != kXPlanes && a.nouts > 0) {
        rows = a.out_rows[g];
        out = a.outs[g];
        obase = 0;
        if (row0 >= rows) return;  // the whole workgroup
    }

    const uint8_t* wrow[NT];
    const float* sp[NWT];
    bool live = true;
#pragma unroll
    for (int i = 0; i < NWT; ++i) {
        live = live && a.w[i][g] != nullptr && a.s[i][g] != nullptr;
        sp[i] = a.s[i][g] + (row0 >> 7) * a.scale_cols;
#pragma unroll
        for (int t = 0; t < TA; ++t) {
            // rows past the end read the last row; their results are dropped
            const int64_t r = min(row0 + 16 * t + li, rows - 1);
            wrow[i * TA + t] =
                a.w[i][g] + (a.tiled ? (r >> 3) * a.nblocks * 1024 + (r & 7) * 128 : r * a.K);
        }
    }
    const int64_t K = a.K;
    const bool ragged = (K & 127) != 0;
    const int nk_all = wave < a.nblocks ? (a.nblocks - 1 - wave) / nw + 1 : 0;

    for (int64_t t0 = static_cast<int64_t>(blockIdx.y) * 16 * TB; t0 < count;
         t0 += static_cast<int64_t>(gridDim.y) * 16 * TB) {
        const char* xrow[TB];
        int64_t lo_off = 0;
        if constexpr (XM == kXPlanes) lo_off = a.xlo - a.x;
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            const int64_t t = min(t0 + 16 * tb + li, count - 1);  // rows past the end repeat the last one
            int64_t r = t;
            if (a.list != nullptr) {
                r = a.list[g * a.list_ld + t];
            } else if (XM == kXPlanes) {
                r = obase + t;
            }
            xrow[tb] = a.x + r * a.x_stride;
        }
        plm_f32x4 acc[2][PL][NT][TB];
        auto pass = [&](auto san) {
            constexpr bool SAN = decltype(san)::value;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int pl = 0; pl < PL; ++pl)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int tb = 0; tb < TB; ++tb) acc[h][pl][t][tb] = plm_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            for (int kb = 0; kb < nk_all; kb += 64) {
                const int nk = min(nk_all - kb, 64);
                float sv[NWT];
#pragma unroll
                for (int n = 0; n < NWT; ++n)
                    sv[n] = plm_gload_f32(sp[n] + wave + static_cast<int64_t>(kb + min(lane, nk - 1)) * nw);
                plm_u32x4 q[P][2][NT];
                XPiece<XB> x[P][2][PL][TB];
                auto issue = [&](int slot, int k) {
                    const int64_t b = wave + static_cast<int64_t>(kb + k) * nw;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        // past the end of a row: its last 16 bytes, masked when used
                        const int64_t off = min(b * 128 + 64 * h + 16 * qd, K - 16);
                        const int64_t woff = a.tiled ? off + (off >> 7) * 896 : off;
#pragma unroll
                        for (int t = 0; t < NT; ++t) q[slot][h][t] = wload16(wrow[t] + woff);
#pragma unroll
                        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                            for (int pl = 0; pl < PL; ++pl)
                                x[slot][h][pl][tb] = load_xpiece<XB>(xrow[tb] + (pl ? lo_off : 0) + off * XE, true);
                    }
                };
                auto compute = [&](int slot, int k) {
                    const int64_t b = wave + static_cast<int64_t>(kb + k) * nw;
                    float sc[NWT];
#pragma unroll
                    for (int n = 0; n < NWT; ++n) sc[n] = lane_value(sv[n], k);
                    // columns past K add nothing
                    auto clip = [](plm_u32x4& v, bool in) { v = in ? v : plm_u32x4{0, 0, 0, 0}; };
                    if (EARLY && ragged) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const bool in = b * 128 + 64 * h + 16 * qd < K;
#pragma unroll
                            for (int t = 0; t < NT; ++t) clip(q[slot][h][t], in);
#pragma unroll
                            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                                for (int i = 0; i < (XB ? 2 : 4); ++i) clip(x[slot][h][0][tb].v[i], in);
                        }
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const bool in = !ragged || b * 128 + 64 * h + 16 * qd < K;
                        plm_bf16x8 a0[NT], a1[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            plm_u32x4 qv = q[slot][h][t];
                            if (!EARLY && ragged) clip(qv, in);
                            weights_to_bf16(SAN ? zero_nan_bytes(qv) : qv, a0[t], a1[t]);
                        }
#pragma unroll
                        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                            for (int pl = 0; pl < PL; ++pl) {
                                XPiece<XB> xv = x[slot][h][pl][tb];
                                if (!EARLY && ragged) {
#pragma unroll
                                    for (int i = 0; i < (XB ? 2 : 4); ++i) clip(xv.v[i], in);
                                }
                                const BOperands<XB, SAN> bo(xv);
#pragma unroll
                                for (int t = 0; t < NT; ++t) {
                                    plm_f32x4 d = mfma_bf16(a0[t], bo.h0, plm_f32x4{0.0f, 0.0f, 0.0f, 0.0f});
                                    d = mfma_bf16(a1[t], bo.h1, d);
                                    if constexpr (!XB) {
                                        d = mfma_bf16(a0[t], bo.l0, d);
                                        d = mfma_bf16(a1[t], bo.l1, d);
                                    }
#pragma unroll
                                    for (int j = 0; j < 4; ++j)
                                        acc[h][pl][t][tb][j] = fmaf(d[j], sc[t / TA], acc[h][pl][t][tb][j]);
                                }
                            }
                    }
                };
                run_pipelined<P>(nk, issue, compute);
            }
        };
        if (live) {
            pass(std::false_type{});
            bool bad = false;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int pl = 0; pl < PL; ++pl)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
#pragma unroll
                        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                bad = bad || acc[h][pl][t][tb][j] != acc[h][pl][t][tb][j];
            // NaN weight bytes count as 0, infinite activations as themselves: the blocks again
            if (__any(bad)) pass(std::true_type{});
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
                plm_f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                if (live) {
                    v = acc[0][0][t][tb] + acc[1][0][t][tb];
                    if constexpr (PL == 2) v = v + (acc[0][1][t][tb] + acc[1][1][t][tb]);
                }
                red[((wave * NT + t) * TB + tb) * 64 + lane] = v;
            }
        __syncthreads();
        // element e of the output tile: weight row fastest (16 rows are 64 bytes of an output row)
        const float* rf = reinterpret_cast<const float*>(red);
        for (int e = threadIdx.x; e < TA * TB * 256; e += blockDim.x) {
            const int r = e & 15, n = (e >> 4) & 15, tt = e >> 8;
            const int ta = tt % TA, tb = tt / TA;
            const int64_t row = row0 + 16 * ta + r, t = t0 + 16 * tb + n;
            if (row >= rows || t >= count) continue;
            float v[NWT];
#pragma unroll
            for (int i = 0; i < NWT; ++i) {
                const int at = (((i * TA + ta) * TB + tb) * 64 + (r >> 2) * 16 + n) * 4 + (r & 3);
                float s = 0.0f;
                for (int w = 0; w < nw; ++w) s += rf[w * NT * TB * 256 + at];
                v[i] = s;
            }
            const int64_t o = (obase + t) * rows + row;
            if constexpr (SILU)
                store_hplanes(a.hhi, a.hlo, o, plm_silu_mul(v[0], v[1]));
            else
                out[o] = v[0];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ (expert, row) pairs
//
// Each expert's weights are read only when a row chose it, and once for 16 of
// its rows: pair_lists_kernel and pair_bases_kernel turn the pairs into lists
// of rows per expert on the device, the gate/up and down launches run each
// expert on its list, and pair_sum_kernel adds each row's results, weighted,
// in ascending order of the experts.

// Slots of the calling workgroup's flagged threads, numbered from `at` in
// thread order; returns the number flagged.  Synchronises the workgroup.
__device__ __forceinline__ int take_slots(bool flag, int at, int* wave_n, int& slot) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
    const uint64_t mask = __ballot(flag);
    if (lane == 0) wave_n[wave] = __popcll(mask);
    __syncthreads();
    int total = 0;
    slot = at + __popcll(mask & ((uint64_t(1) << lane) - 1));
    for (int w = 0; w < waves; ++w) {
        if (w < wave) slot += wave_n[w];
        total += wave_n[w];
    }
    __syncthreads();
    return total;
}

constexpr int kPairThreads = 256;

// Workgroup e: expert e's route weight of every row (the sum of its pairs'
// weights in pair order; rows without one 0), the ascending list of the rows
// whose weight is not 0, and each row's place in it (-1: not in it).
// Workgroup 0 also counts the pairs with an index out of range.
__global__ __launch_bounds__(kPairThreads) void pair_lists_kernel(const int64_t* __restrict__ items,
                                                                  const int64_t* __restrict__ rows,
                                                                  const float* __restrict__ w, int64_t pairs,
                                                                  int64_t experts, int64_t batch, float* route,
                                                                  int* place, int* list, int* count, int* bad) {
    __shared__ int wave_n[kPairThreads / 64];
    __shared__ int64_t s_row[kPairThreads];
    __shared__ float s_w[kPairThreads];
    const int tid = threadIdx.x;
    const int64_t e = blockIdx.x;
    float* my_route = route + e * batch;
    int* my_place = place + e * batch;
    int* my_list = list + e * batch;
    for (int64_t r = tid; r < batch; r += kPairThreads) my_route[r] = 0.0f;
    int nbad = 0;
    __syncthreads();
    for (int64_t p0 = 0; p0 < pairs; p0 += kPairThreads) {
        const int64_t p = p0 + tid;
        const int64_t it = p < pairs ? items[p] : 0, r = p < pairs ? rows[p] : 0;
        const bool row_ok = r >= 0 && r < batch;
        nbad += p < pairs && (it < 0 || it >= experts || !row_ok);
        int slot;
        const bool hit = p < pairs && it == e && row_ok;
        const int n = take_slots(hit, 0, wave_n, slot);
        if (n == 0) continue;
        if (hit) {
            s_row[slot] = r;
            s_w[slot] = w[p];
        }
        __syncthreads();
        if (tid < n) {
            // the first pair of its row adds every pair of that row, in order
            const int64_t row = s_row[tid];
            bool first = true;
            for (int i = 0; i < tid; ++i) first = first && s_row[i] != row;
            if (first) {
                float v = my_route[row];
                for (int i = tid; i < n; ++i)
                    if (s_row[i] == row) v += s_w[i];
                my_route[row] = v;
            }
        }
        __syncthreads();
    }
    int total = 0;
    for (int64_t r0 = 0; r0 < batch; r0 += kPairThreads) {
        const int64_t r = r0 + tid;
        const bool in = r < batch && my_route[r] != 0.0f;
        int slot;
        const int n = take_slots(in, total, wave_n, slot);
        if (r < batch) my_place[r] = in ? slot : -1;
        if (in) my_list[slot] = static_cast<int>(r);
        total += n;
    }
    if (tid == 0) count[e] = total;
    if (bad != nullptr && e == 0) {
        __shared__ int sum;
        if (tid == 0) sum = 0;
        __syncthreads();
        if (nbad) atomicAdd(&sum, nbad);
        __syncthreads();
        if (tid == 0) *bad = sum;
    }
}

// base[e] = count[0] + ... + count[e - 1].  One wave.
__global__ __launch_bounds__(64) void pair_bases_kernel(const int* __restrict__ count, int* __restrict__ base,
                                                        int64_t experts) {
    const int lane = threadIdx.x;
    int carry = 0;
    for (int64_t e0 = 0; e0 < experts; e0 += 64) {
        const int64_t e = e0 + lane;
        const int n = e < experts ? count[e] : 0;
        int v = n;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(v, off);
            if (lane >= off) v += up;
        }
        if (e < experts) base[e] = carry + v - n;
        carry += __shfl(v, 63);
    }
}

// Workgroup (row m, 1024 columns): the row's experts in ascending order.
__global__ __launch_bounds__(kPairThreads) void pair_sum_kernel(const float* __restrict__ part,
                                                                const float* __restrict__ route,
                                                                const int* __restrict__ place,
                                                                const int* __restrict__ base, int64_t experts,
                                                                int64_t batch, int64_t hid, float* __restrict__ out) {
    __shared__ int wave_n[kPairThreads / 64];
    __shared__ int s_slot[kPairThreads];
    __shared__ float s_w[kPairThreads];
    const int64_t m = blockIdx.x;
    const int64_t col = (static_cast<int64_t>(blockIdx.y) * kPairThreads + threadIdx.x) * 4;
    plm_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int64_t e0 = 0; e0 < experts; e0 += kPairThreads) {
        const int64_t e = e0 + threadIdx.x;
        const int at = e < experts ? place[e * batch + m] : -1;
        int slot;
        const int n = take_slots(at >= 0, 0, wave_n, slot);
        if (at >= 0) {
            s_slot[slot] = base[e] + at;
            s_w[slot] = route[e * batch + m];
        }
        __syncthreads();
        if (col < hid)
            for (int i = 0; i < n; ++i) {
                const plm_f32x4 v = *reinterpret_cast<const plm_f32x4*>(part + s_slot[i] * hid + col);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = fmaf(v[j], s_w[i], acc[j]);
            }
        __syncthreads();
    }
    if (col < hid)
#pragma unroll
        for (int j = 0; j < 4; ++j) out[m * hid + col + j] = acc[j];
}

// ------------------------------------------------------------------ prompt chunks
//
// fp8_panel_kernel: a workgroup of 4 WR waves owns 64 WR weight rows and 8
// column tiles of 16 (128 bf16 activation rows, or 64 rows as hi and lo).
// The block's weights (as bytes, NaN bytes zeroed) and activations go through
// LDS in the order the MFMA operands are read, double buffered, the next
// block's loads in flight meanwhile: a weight byte is read once per 64 to 128
// activation rows and an activation once per 64 to 128 weight rows.  Wave
// (wr, wc) computes 32 rows by 4 column tiles.  The K blocks run in the order
// of the skinny kernel's waves: the blocks of one wave into the two halves'
// accumulators, which are then added to the total, so the sums are the same
// bits.
//
// What bounds it: a wave's own instructions (at one to two waves per SIMD
// conversions, scaling FMAs, MFMAs and LDS reads hardly overlap: of the busy
// cycles of the bf16 linear below the vector units issue in 46 %, the matrix
// cores and the LDS work in 25 % each; more workgroups per compute unit, deeper
// prefetch or single buffers changed nothing).  24576x1536 at 509 bf16 rows:
// 289 us with the skinny kernel, 75 here (510 TFLOP/s) and 5 for packing; the
// 7168 / 2048 MLP at 256 fp32 rows 251 -> 107 us (gate + up 73, down 38).
//
// The activations come packed ([block][column tile][half][piece][lane]
// [8 values], kTileBytes per column tile and block) by fp8_pack_rows_kernel,
// or from the gate/up launch's epilogue.  Rows past m hold anything (their
// columns are dropped); columns past K are zero.

using plm::kPanelCols;
using plm::panel_tiles;
constexpr int kTileBytes = 4096;   // one column tile of one block

struct PanelArgs {
    const uint8_t* w[2];
    const float* s[2];
    const char* x;
    float* out;
    char* xout;  // SILU: the packed hi / lo columns of silu(gate) * up
    int64_t rows;
    int64_t K;
    int64_t scale_cols;
    int64_t m;
    int nblocks;
    int waves;      // K slots
    int row_tiles;  // workgroups along the rows
    int col_tiles;  // workgroups along the activation rows
    int out_tiles;  // SILU: column tiles of xout
    int x_tiles;    // column tiles of x
    int tiled;
    // The K slots dealt to `splits` workgroups a tile (slot k to part k %
    // splits): every slot's sums go to part[slot][m][part_ld] and a second
    // kernel adds them in order.  1: the workgroup adds them itself.
    int splits;
    float* part;
    int64_t part_ld;
};

// Byte offset of column `col` of activation row `li` of column tile `tile`.
__device__ __forceinline__ int64_t packed_at(int64_t col, int tiles, int tile, int li) {
    return ((col >> 7) * tiles + tile) * kTileBytes + ((col >> 6) & 1) * 2048 + ((col >> 3) & 1) * 1024 +
           (((col >> 4) & 3) * 16 + li) * 16 + (col & 7) * 2;
}

// WR: 64 weight rows each (two wave rows of 32); MODE: bf16 activations
// (kXBf16), fp32 ones as hi and lo in one chain (kXF32), or planes with
// accumulators of their own (kXPlanes).
template <int WR, bool SILU, int MODE, bool SPLIT>
__global__ __launch_bounds__(256 * WR, 2) void fp8_panel_kernel(const PanelArgs a) {
    constexpr int NW = 4 * WR;                    // waves: 2 WR along the rows, 2 along the columns
    constexpr int CT = MODE == kXBf16 ? 4 : 2;    // token tiles per wave
    constexpr int PL = MODE == kXPlanes ? 2 : 1;  // accumulator planes
    constexpr int ABYTES = 4 * WR * 2048;         // a block's weights
    constexpr int XBYTES = kPanelCols * kTileBytes;
    constexpr int XL = XBYTES / (NW * 1024);      // activation loads per lane and block
    constexpr int DEPTH = WR == 1 && MODE != kXPlanes ? 2 : 1;  // blocks in flight in registers
    constexpr int STAGES = MODE == kXPlanes ? 1 : 2;            // blocks in LDS
    extern __shared__ char panel[];               // [STAGES][ABYTES + XBYTES]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, li = lane & 15, qd = lane >> 4;
    const int wr = wave / 2, wc = wave % 2;
    // workgroup -> tile: the column tiles of a row tile follow each other on one XCD
    const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
    const int rt = (seq / a.col_tiles) * 8 + xcd, ct = seq % a.col_tiles;
    if (rt >= a.row_tiles) return;
    constexpr int ROWS = SILU ? 32 * WR : 64 * WR;  // rows of one weight
    const int64_t row0 = static_cast<int64_t>(rt) * ROWS;
    const int64_t K = a.K;
    const int nb = a.nblocks, nw = a.waves;

    // the 16-row tile this wave loads: tiles 2 wr + t are wave row wr's; SILU: t = 0 gate, 1 up
    const int64_t my_row = min(row0 + (SILU ? 16 * (wave / 2) : 16 * wave) + li, a.rows - 1);  // past the end: dropped
    const uint8_t* wrow = (SILU && (wave & 1) ? a.w[1] : a.w[0]) +
                          (a.tiled ? (my_row >> 3) * nb * 1024 + (my_row & 7) * 128 : my_row * K);
    const float* sp[2];
    sp[0] = a.s[0] + (row0 >> 7) * a.scale_cols;
    sp[1] = SILU ? a.s[1] + (row0 >> 7) * a.scale_cols : sp[0];
    const char* xsrc = a.x + static_cast<int64_t>(ct) * XBYTES + threadIdx.x * 16;
    const int64_t xstep = static_cast<int64_t>(a.x_tiles) * kTileBytes;

    // DEPTH blocks in flight in registers; the scales by vector loads: a
    // scalar load in flight would hold up every LDS read (they share a counter
    // and scalar loads return out of order)
    plm_u32x4 wq[DEPTH][2], xq[DEPTH][XL];
    float snext[DEPTH][2];
    int vzero = 0;
    asm("" : "+v"(vzero));
    // the block after b in the order of this workgroup's K slots (nb: none)
    const int first = SPLIT ? blockIdx.y : 0, step = SPLIT ? a.splits : 1;
    auto after = [&](int b) { return b + nw < nb ? b + nw : (b % nw + step < nw ? b % nw + step : nb); };
    int fb;  // the next block to fetch
    auto fetch = [&](int u) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            // past the end of a row: its last 16 bytes, against zero activations
            const int64_t off = min(static_cast<int64_t>(fb) * 128 + 64 * h + 16 * qd, K - 16);
            wq[u][h] = xload16(wrow + (a.tiled ? off + (off >> 7) * 896 : off));
        }
#pragma unroll
        for (int i = 0; i < XL; ++i) xq[u][i] = xload16(xsrc + fb * xstep + i * NW * 1024);
        snext[u][0] = plm_gload_f32(sp[0] + fb + vzero);
        if (SILU) snext[u][1] = plm_gload_f32(sp[1] + fb + vzero);
        fb = after(fb);
    };
    // D: lane (activation row li, weight rows 4 qd + j)
    auto token_tile = [&](int c) { return (ct * kPanelCols + wc * 4) / (MODE == kXBf16 ? 1 : 2) + c; };
    // 4 floats at `row` of an output row of a.rows, the last of them perhaps past its end
    auto store_row = [&](float* out, int64_t row, plm_f32x4 v) {
        if (row + 4 <= a.rows && (reinterpret_cast<uintptr_t>(out + row) & 15) == 0) {
            *reinterpret_cast<plm_f32x4*>(out + row) = v;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (row + j < a.rows) out[row + j] = v[j];
        }
    };
    plm_f32x4 acc[2][PL][2][CT], total[2][CT];
    bool bad = false;  // a NaN among the sums of an activation row
    auto store_part = [&](int slot, int t, int c, plm_f32x4 v) {
        const int64_t t_row = static_cast<int64_t>(token_tile(c)) * 16 + li;
        if (t_row >= a.m) return;
#pragma unroll
        for (int j = 0; j < 4; ++j) bad = bad || v[j] != v[j];
        // SILU: gate in columns 0 .., up in part_ld / 2 ..
        store_row(a.part + (slot * a.m + t_row) * a.part_ld + (SILU && t ? a.part_ld / 2 : 0),
                  row0 + (SILU ? 16 * wr : 32 * wr + 16 * t) + 4 * qd, v);
    };
    int stage = 0, cb;  // cb: the block being computed
    // A block: its operands to LDS, the loads of the block DEPTH further, its products.
    auto block = [&](int u, bool zero_nans) {
        char* as = panel + stage * (ABYTES + XBYTES);
        char* xs = as + ABYTES;
        if (STAGES == 1) __syncthreads();  // the last block's reads
#pragma unroll
        for (int h = 0; h < 2; ++h)
            *reinterpret_cast<plm_u32x4*>(as + (wave * 2 + h) * 1024 + lane * 16) =
                zero_nans ? zero_nan_bytes(wq[u][h]) : wq[u][h];
#pragma unroll
        for (int i = 0; i < XL; ++i)
            *reinterpret_cast<plm_u32x4*>(xs + i * NW * 1024 + threadIdx.x * 16) = xq[u][i];
        float sc[2];
        sc[0] = lane_value(snext[u][0], 0);
        sc[1] = SILU ? lane_value(snext[u][1], 0) : sc[0];
        if (cb < nw) {  // a slot's first block
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int pl = 0; pl < PL; ++pl)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int c = 0; c < CT; ++c) acc[h][pl][t][c] = plm_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        if (fb < nb) fetch(u);
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            plm_bf16x8 a0[2], a1[2];
#pragma unroll
            for (int t = 0; t < 2; ++t)
                weights_to_bf16(*reinterpret_cast<const plm_u32x4*>(as + ((wr * 2 + t) * 2 + h) * 1024 + lane * 16),
                                a0[t], a1[t]);
            auto operand = [&](int c, int p) {  // of the wave's column tile c, piece p
                return *reinterpret_cast<const plm_bf16x8*>(xs + (wc * 4 + c) * kTileBytes + h * 2048 + p * 1024 +
                                                            lane * 16);
            };
            auto add = [&](plm_f32x4& to, plm_f32x4 d, float f) {
#pragma unroll
                for (int j = 0; j < 4; ++j) to[j] = fmaf(d[j], f, to[j]);
            };
            const plm_f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (MODE == kXF32) {
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    const plm_bf16x8 h0 = operand(2 * c, 0), h1 = operand(2 * c, 1);
                    const plm_bf16x8 l0 = operand(2 * c + 1, 0), l1 = operand(2 * c + 1, 1);
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        plm_f32x4 d = mfma_bf16(a0[t], h0, none);
                        d = mfma_bf16(a1[t], h1, d);
                        d = mfma_bf16(a0[t], l0, d);
                        d = mfma_bf16(a1[t], l1, d);
                        add(acc[h][0][t][c], d, sc[SILU ? t : 0]);
                    }
                }
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const plm_bf16x8 b0 = operand(c, 0), b1 = operand(c, 1);
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        plm_f32x4 d = mfma_bf16(a0[t], b0, none);
                        d = mfma_bf16(a1[t], b1, d);
                        add(MODE == kXPlanes ? acc[h][c % PL][t][c / 2] : acc[h][0][t][c % CT], d, sc[SILU ? t : 0]);
                    }
                }
            }
        }
        if (cb + nw >= nb) {  // the slot's last block
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    plm_f32x4 v = acc[0][0][t][c] + acc[1][0][t][c];
                    if constexpr (PL == 2) v = v + (acc[0][1][t][c] + acc[1][1][t][c]);
                    if constexpr (SPLIT)
                        store_part(cb % nw, t, c, v);
                    else
                        total[t][c] = total[t][c] + v;
                }
        }
        if (STAGES == 2) stage ^= 1;
        cb = after(cb);
    };
    auto pass = [&](bool zero_nans) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int c = 0; c < CT; ++c) total[t][c] = plm_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        fb = cb = first;
#pragma unroll
        for (int u = 0; u < DEPTH; ++u)
            if (fb < nb) fetch(u);
        while (cb < nb) {
#pragma unroll
            for (int u = 0; u < DEPTH; ++u)
                if (cb < nb) block(u, zero_nans);
        }
    };
    pass(false);
    if constexpr (!SPLIT) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    bad = bad || (total[t][c][j] != total[t][c][j] && token_tile(c) * 16 + li < a.m);
    }
    // NaN weight bytes count as 0: the blocks again (rows without one come out the same)
    if (__syncthreads_or(bad)) pass(true);
    if constexpr (SPLIT) return;

#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int tile = token_tile(c);
        const int64_t t_row = static_cast<int64_t>(tile) * 16 + li;
        if constexpr (SILU) {
            if (tile >= a.out_tiles / 2) continue;
            // 4 of the 16 columns (row0 + 16 wr ..) of the down phase's activations
            const int64_t col = row0 + 16 * wr + 4 * qd;
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                split_f32<true>(__float_as_uint(plm_silu_mul(total[0][c][j], total[1][c][j])), hi[j], lo[j]);
                if (col + j >= a.rows) hi[j] = lo[j] = 0u;
            }
            char* o = a.xout + packed_at(col, a.out_tiles, 2 * tile, li);
            *reinterpret_cast<uint2*>(o) = make_uint2(hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16));
            *reinterpret_cast<uint2*>(o + kTileBytes) = make_uint2(lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16));
        } else if (t_row < a.m) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
                store_row(a.out + t_row * a.rows, row0 + 32 * wr + 16 * t + 4 * qd, total[t][c]);
        }
    }
}

// The slots' sums of a split launch, added in order.
__global__ __launch_bounds__(256) void fp8_panel_sum_kernel(const float* __restrict__ part, int slots, int64_t n,
                                                            float* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    float v = 0.0f;
    for (int k = 0; k < slots; ++k) v += part[k * n + i];
    out[i] = v;
}

// The same for gate and up (rows [gate | up] of ld columns), with the SiLU
// epilogue: one thread per activation row and 8 columns of the packed
// intermediate.
__global__ __launch_bounds__(256) void fp8_panel_silu_kernel(const float* __restrict__ part, int slots, int64_t m,
                                                             int64_t ld, int64_t rows, char* __restrict__ xout,
                                                             int out_tiles, int64_t pieces) {
    const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t t_row = id / pieces, col = (id - t_row * pieces) * 8;
    if (t_row >= m) return;
    float g[8], u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) g[j] = u[j] = 0.0f;
    if (col < rows)  // rows is a multiple of 16
        for (int k = 0; k < slots; ++k) {
            const float* p = part + (k * m + t_row) * ld + col;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                g[j] += p[j];
                u[j] += p[ld / 2 + j];
            }
        }
    uint32_t hi[8], lo[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        split_f32<true>(__float_as_uint(plm_silu_mul(g[j], u[j])), hi[j], lo[j]);
        if (col >= rows) hi[j] = lo[j] = 0u;
    }
    char* o = xout + packed_at(col, out_tiles, static_cast<int>(t_row >> 4) * 2, static_cast<int>(t_row & 15));
    *reinterpret_cast<uint4*>(o) = make_uint4(hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16), hi[4] | (hi[5] << 16),
                                              hi[6] | (hi[7] << 16));
    *reinterpret_cast<uint4*>(o + kTileBytes) = make_uint4(lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16),
                                                           lo[4] | (lo[5] << 16), lo[6] | (lo[7] << 16));
}

// Activation rows packed for fp8_panel_kernel: one wave per (block, half,
// token tile); fp32 rows as the column tiles 2 t (hi) and 2 t + 1 (lo).
template <bool XB>
__global__ __launch_bounds__(256) void fp8_pack_rows_kernel(const char* __restrict__ x, char* __restrict__ out,
                                                            int64_t m, int64_t K, int64_t stride, int token_tiles,
                                                            int x_tiles, int nblocks) {
    const int64_t id = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int h = id & 1;
    const int64_t tile = (id >> 1) % token_tiles, b = (id >> 1) / token_tiles;
    if (b >= nblocks) return;
    const int64_t row = tile * 16 + (lane & 15), col = b * 128 + 64 * h + 16 * (lane >> 4);
    if (row >= m) return;
    plm_u32x4 hi[2] = {}, lo[2] = {};
    if (col < K) {  // K is a multiple of 16
        const char* src = x + row * stride + col * (XB ? 2 : 4);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if constexpr (XB) {
                hi[p] = xload16(src + 16 * p);
            } else {
                plm_bf16x8 vh, vl;
                split8<true>(xload16(src + 32 * p), xload16(src + 32 * p + 16), vh, vl);
                hi[p] = __builtin_bit_cast(plm_u32x4, vh);
                lo[p] = __builtin_bit_cast(plm_u32x4, vl);
            }
        }
    }
    char* o = out + (b * x_tiles + tile * (XB ? 1 : 2)) * kTileBytes + h * 2048 + lane * 16;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        *reinterpret_cast<plm_u32x4*>(o + p * 1024) = hi[p];
        if (!XB) *reinterpret_cast<plm_u32x4*>(o + kTileBytes + p * 1024) = lo[p];
    }
}

int64_t panel_bytes(int64_t m, int64_t K, bool one_plane) {
    return plm::ceil_div(K, 128) * panel_tiles(m, one_plane) * kTileBytes;
}

int pack_rows(const float* x, const uint16_t* xb, int64_t m, int64_t K, int64_t stride, char* out, hipStream_t st) {
    const int token_tiles = static_cast<int>(plm::ceil_div(m, 16));
    const int nb = static_cast<int>(plm::ceil_div(K, 128));
    const dim3 grid(static_cast<unsigned>(plm::ceil_div(static_cast<int64_t>(nb) * token_tiles * 2, 4)));
    if (xb != nullptr)
        hipLaunchKernelGGL((fp8_pack_rows_kernel<true>), grid, dim3(256), 0, st, reinterpret_cast<const char*>(xb), out,
                           m, K, stride * 2, token_tiles, panel_tiles(m, true), nb);
    else
        hipLaunchKernelGGL((fp8_pack_rows_kernel<false>), grid, dim3(256), 0, st, reinterpret_cast<const char*>(x), out,
                           m, K, stride * 4, token_tiles, panel_tiles(m, false), nb);
    return plm::check_launch("fp8 pack rows");
}

template <int WR, bool SILU, int MODE, bool SPLIT = false>
int launch_panel(const PanelArgs& args, hipStream_t st) {
    PanelArgs a = args;
    // SILU: whole 128-column blocks of the down phase's activations
    a.row_tiles = static_cast<int>(SILU ? plm::ceil_div(a.rows, 128) * 128 / (32 * WR) : plm::ceil_div(a.rows, 64 * WR));
    a.col_tiles = a.x_tiles / kPanelCols;
    const unsigned grid = static_cast<unsigned>(plm::ceil_div(a.row_tiles, 8) * 8 * a.col_tiles);
    constexpr int kLds = (MODE == kXPlanes ? 1 : 2) * (4 * WR * 2048 + kPanelCols * kTileBytes);
    const void* fn = reinterpret_cast<const void*>(&fp8_panel_kernel<WR, SILU, MODE, SPLIT>);
    int code = plm::allow_large_lds(fn, kLds);
    if (code != 0) return code;
    hipLaunchKernelGGL((fp8_panel_kernel<WR, SILU, MODE, SPLIT>), dim3(grid, static_cast<unsigned>(a.splits)),
                       dim3(256 * WR), kLds, st, a);
    code = plm::check_launch("fp8 panel kernel");
    if (code != 0 || !SPLIT) return code;
    if (SILU) {
        const int64_t pieces = plm::ceil_div(a.rows, 128) * 16;
        hipLaunchKernelGGL(fp8_panel_silu_kernel, dim3(static_cast<unsigned>(plm::ceil_div(a.m * pieces, 256))),
                           dim3(256), 0, st, a.part, a.waves, a.m, a.part_ld, a.rows, a.xout, a.out_tiles, pieces);
    } else {
        const int64_t n = a.m * a.rows;
        hipLaunchKernelGGL(fp8_panel_sum_kernel, dim3(static_cast<unsigned>(plm::ceil_div(n, 256))), dim3(256), 0, st,
                           a.part, a.waves, n, a.out);
    }
    return plm::check_launch("fp8 panel sum");
}

// Floats of the slots' sums.
int64_t panel_part(int64_t rows, bool silu, int x_tiles, int waves, int64_t m) {
    const int splits = plm::panel_plan(rows, silu, x_tiles, waves, plm::cu_count()).splits;
    return splits == 1 ? 0 : waves * m * rows * (silu ? 2 : 1);
}

template <bool SILU, int MODE>
int launch_panel_rows(const PanelArgs& args, float* part, hipStream_t st) {
    PanelArgs a = args;
    const plm::PanelPlan plan = plm::panel_plan(a.rows, SILU, a.x_tiles, a.waves, plm::cu_count());
    a.splits = plan.splits;
    a.part = part;
    a.part_ld = a.rows * (SILU ? 2 : 1);
    if (plan.wr == 2) return launch_panel<2, SILU, MODE>(a, st);
    return plan.splits == 1 ? launch_panel<1, SILU, MODE>(a, st) : launch_panel<1, SILU, MODE, true>(a, st);
}

PanelArgs panel_args(const plm::BatchRows& p, const char* x, int x_tiles, int64_t m) {
    PanelArgs a;
    std::memset(&a, 0, sizeof(a));
    for (int i = 0; i < (p.hhi != nullptr ? 2 : 1); ++i) {
        a.w[i] = p.w[i][0];
        a.s[i] = p.s[i][0];
    }
    a.x = x;
    a.out = p.out;
    a.rows = p.rows;
    a.K = p.K;
    a.scale_cols = p.scale_cols;
    a.m = m;
    a.nblocks = static_cast<int>(plm::ceil_div(p.K, 128));
    a.waves = p.waves;
    a.x_tiles = x_tiles;
    a.tiled = p.tiled ? 1 : 0;
    return a;
}

template <int TA, int TB, int P, int NWT, bool SILU, int XM, int MAXW>
int launch(const plm::BatchRows& p, const BatchArgs& args, int chunks, hipStream_t st) {
    BatchArgs a = args;
    a.tiles = static_cast<int>(plm::ceil_div(p.rows, 16 * TA));
    const dim3 grid(static_cast<unsigned>(a.tiles) * p.ngroups, static_cast<unsigned>(chunks));
    const size_t lds = static_cast<size_t>(p.waves) * NWT * TA * TB * 1024;
    static_assert(MAXW * NWT * TA * TB * 1024 <= 65536, "the waves' sums fit 64 KB");
    hipLaunchKernelGGL((fp8_batch_kernel<TA, TB, P, NWT, SILU, XM, MAXW>), grid, dim3(p.waves * plm::kWave), lds, st,
                       a);
    return plm::check_launch("fp8 batch kernel");
}

}  // namespace

int plm::fp8_batch_rows(const BatchRows& p, hipStream_t st) {
    BatchArgs a;
    std::memset(&a, 0, sizeof(a));
    const bool silu = p.hhi != nullptr;
    for (int i = 0; i < (silu ? 2 : 1); ++i)
        for (int g = 0; g < p.ngroups; ++g) {
            a.w[i][g] = p.w[i][g];
            a.s[i][g] = p.s[i][g];
        }
    const int xm = p.xhi != nullptr ? kXPlanes : (p.xb != nullptr ? kXBf16 : kXF32);
    a.x = xm == kXPlanes ? reinterpret_cast<const char*>(p.xhi)
                         : (xm == kXBf16 ? reinterpret_cast<const char*>(p.xb) : reinterpret_cast<const char*>(p.x));
    a.xlo = reinterpret_cast<const char*>(p.xlo);
    a.x_stride = p.x_stride * (xm == kXF32 ? 4 : 2);
    a.out = p.out;
    a.hhi = p.hhi;
    a.hlo = p.hlo;
    a.rows = p.rows;
    a.K = p.K;
    a.scale_cols = p.scale_cols;
    a.m = p.m;
    a.list_ld = p.groups.list_ld;
    a.count = p.groups.count;
    a.base = p.groups.base;
    a.list = p.groups.list;
    a.nblocks = static_cast<int>(plm::ceil_div(p.K, 128));
    a.tiled = p.tiled ? 1 : 0;
    if (p.outs[0] != nullptr) {
        if (p.ngroups > kBatchOuts) return plm::fail(-2, "1..%d weights per call", kBatchOuts);
        a.nouts = p.ngroups;
        for (int g = 0; g < p.ngroups; ++g) {
            a.outs[g] = p.outs[g];
            a.out_rows[g] = p.out_rows[g];
        }
    }
    const bool grouped = p.groups.count != nullptr;
    const int64_t m = p.m;
    auto chunks = [&](int tb) { return grouped ? 1 : static_cast<int>(plm::ceil_div(m, 16 * tb)); };
    if (silu) {
        if (grouped || m <= 16)
            return xm == kXBf16 ? launch<1, 1, 2, 2, true, kXBf16, 4>(p, a, chunks(1), st)
                                : launch<1, 1, 2, 2, true, kXF32, 4>(p, a, chunks(1), st);
        return xm == kXBf16 ? launch<1, 2, 2, 2, true, kXBf16, 4>(p, a, chunks(2), st)
                            : launch<1, 2, 1, 2, true, kXF32, 4>(p, a, chunks(2), st);
    }
    if (xm == kXPlanes) return launch<2, 1, 1, 1, false, kXPlanes, 16>(p, a, chunks(1), st);
    // 16 weight rows a workgroup while that still leaves at most one for each
    // compute unit, else 32: a workgroup's time is its chain of K blocks, and
    // half of the rows take less than half of the work (2048x7168 at 9 and 16
    // bf16 rows, us: 15.7 and 18.2 -> 11.4 and 13.6, at 64 37.9 -> 32.8; fp32
    // 19.8 and 25.1 -> 15.4 and 20.7).  Past one round the wider tile wins:
    // 7168x2048 at 16 rows 8.3 against 9.5, 4096x7168 at 65 39 against 48.
    const int tb = m <= 16 ? 1 : (m <= 32 || xm == kXF32 ? 2 : 4);
    int64_t narrow = 0;
    for (int g = 0; g < p.ngroups; ++g) narrow += plm::ceil_div(p.outs[0] != nullptr ? p.out_rows[g] : p.rows, 16);
    if (narrow * chunks(tb) <= plm::cu_count()) {
        if (xm == kXBf16)
            return tb == 1 ? launch<1, 1, 2, 1, false, kXBf16, 8>(p, a, chunks(1), st)
                           : (tb == 2 ? launch<1, 2, 2, 1, false, kXBf16, 8>(p, a, chunks(2), st)
                                      : launch<1, 4, 2, 1, false, kXBf16, 8>(p, a, chunks(4), st));
        return tb == 1 ? launch<1, 1, 2, 1, false, kXF32, 8>(p, a, chunks(1), st)
                       : launch<1, 2, 2, 1, false, kXF32, 8>(p, a, chunks(2), st);
    }
    if (xm == kXBf16)
        return tb == 1 ? launch<2, 1, 2, 1, false, kXBf16, 8>(p, a, chunks(1), st)
                       : (tb == 2 ? launch<2, 2, 2, 1, false, kXBf16, 8>(p, a, chunks(2), st)
                                  : launch<2, 4, 1, 1, false, kXBf16, 8>(p, a, chunks(4), st));
    return tb == 1 ? launch<2, 1, 2, 1, false, kXF32, 8>(p, a, chunks(1), st)
                   : launch<2, 2, 1, 1, false, kXF32, 8>(p, a, chunks(2), st);
}

namespace {

// Activation rows of a call beyond kPanelPass go in passes over the weights, so
// that its packed copy stays a bounded part of the thread's scratch (268 MB for
// 16384 fp32 columns): one read of a weight in 4096 rows is nothing.
constexpr int64_t kPanelPass = 4096;

template <class Pass>
int in_passes(int64_t m, Pass pass) {
    int code = 0;
    for (int64_t m0 = 0; m0 < m && code == 0; m0 += kPanelPass) code = pass(m0, std::min(kPanelPass, m - m0));
    return code;
}

int panel_linear_rows(const plm::BatchRows& p, int64_t m0, int64_t m, hipStream_t st) {
    const bool bf16 = p.xb != nullptr;
    const int tiles = panel_tiles(m, bf16);
    const int64_t first = panel_bytes(m, p.K, bf16);
    int64_t part = 0;
    for (int i = 0; i < p.ngroups; ++i) part = std::max(part, panel_part(p.out_rows[i], false, tiles, p.waves, m));
    char* x = static_cast<char*>(plm::workspace(static_cast<size_t>(first + part * 4)));
    if (x == nullptr) return -3;
    float* sums = reinterpret_cast<float*>(x + first);
    const int64_t skip = m0 * p.x_stride;
    int code = pack_rows(bf16 ? nullptr : p.x + skip, bf16 ? p.xb + skip : nullptr, m, p.K, p.x_stride, x, st);
    for (int i = 0; i < p.ngroups && code == 0; ++i) {
        PanelArgs a = panel_args(p, x, tiles, m);
        a.w[0] = p.w[0][i];
        a.s[0] = p.s[0][i];
        a.out = p.outs[i] + m0 * p.out_rows[i];
        a.rows = p.out_rows[i];
        code = bf16 ? launch_panel_rows<false, kXBf16>(a, sums, st) : launch_panel_rows<false, kXF32>(a, sums, st);
    }
    return code;
}

int panel_mlp_rows(const plm::BatchRows& gate_up, const plm::BatchRows& down, int64_t m0, int64_t m, hipStream_t st) {
    const bool bf16 = gate_up.xb != nullptr;
    const int tiles = panel_tiles(m, bf16), out_tiles = panel_tiles(m, false);
    const int64_t first = panel_bytes(m, gate_up.K, bf16), second = panel_bytes(m, down.K, false);
    const int64_t part = std::max(panel_part(gate_up.rows, true, tiles, gate_up.waves, m),
                                  panel_part(down.rows, false, out_tiles, down.waves, m));
    char* x = static_cast<char*>(plm::workspace(static_cast<size_t>(first + second + part * 4)));
    if (x == nullptr) return -3;
    float* sums = reinterpret_cast<float*>(x + first + second);
    const int64_t skip = m0 * gate_up.x_stride;
    int code = pack_rows(bf16 ? nullptr : gate_up.x + skip, bf16 ? gate_up.xb + skip : nullptr, m, gate_up.K,
                         gate_up.x_stride, x, st);
    if (code != 0) return code;
    PanelArgs a = panel_args(gate_up, x, tiles, m);
    for (int i = 0; i < 2; ++i) {
        a.w[i] = gate_up.w[i][0];
        a.s[i] = gate_up.s[i][0];
    }
    a.xout = x + first;
    a.out_tiles = out_tiles;
    code = bf16 ? launch_panel_rows<true, kXBf16>(a, sums, st) : launch_panel_rows<true, kXF32>(a, sums, st);
    if (code != 0) return code;
    PanelArgs d = panel_args(down, x + first, out_tiles, m);
    d.out += m0 * down.rows;
    return launch_panel_rows<false, kXPlanes>(d, sums, st);
}

}  // namespace

int plm::fp8_panel_linear(const BatchRows& p, hipStream_t st) {
    return in_passes(p.m, [&](int64_t m0, int64_t m) { return panel_linear_rows(p, m0, m, st); });
}

int plm::fp8_panel_mlp(const BatchRows& gate_up, const BatchRows& down, hipStream_t st) {
    return in_passes(gate_up.m, [&](int64_t m0, int64_t m) { return panel_mlp_rows(gate_up, down, m0, m, st); });
}

int plm::fp8_batch_pairs(const PairProblem& p, hipStream_t st) {
    const int64_t cells = p.experts * p.batch;
    const int64_t slots = std::min(p.pairs, cells);  // rows of the lists, all experts together
    if (p.experts > 0x7FFFFFFF / 2 || p.batch > 0x7FFFFFFF / 2 || slots > 0x7FFFFFFF / 2)
        return plm::fail(-2, "too many pairs");
    // workspace: route f32, place, list i32 [experts][batch] | count, base i32 [experts] | planes | results
    const int64_t sizes[] = {cells * 4, cells * 4, cells * 4, p.experts * 4, p.experts * 4, slots * p.inter * 4,
                             slots * p.hid * 4};
    constexpr int kBufs = static_cast<int>(sizeof(sizes) / sizeof(sizes[0]));
    int64_t off[kBufs], total = 0;
    for (int i = 0; i < kBufs; ++i) {
        off[i] = total;
        total += plm::ceil_div(sizes[i], 256) * 256;
    }
    char* ws = static_cast<char*>(plm::workspace(static_cast<size_t>(total)));
    if (ws == nullptr) return -3;
    float* route = reinterpret_cast<float*>(ws + off[0]);
    int* place = reinterpret_cast<int*>(ws + off[1]);
    int* list = reinterpret_cast<int*>(ws + off[2]);
    int* count = reinterpret_cast<int*>(ws + off[3]);
    int* base = reinterpret_cast<int*>(ws + off[4]);
    uint16_t* planes = reinterpret_cast<uint16_t*>(ws + off[5]);
    float* part = reinterpret_cast<float*>(ws + off[6]);
    hipLaunchKernelGGL(pair_lists_kernel, dim3(static_cast<unsigned>(p.experts)), dim3(kPairThreads), 0, st, p.items,
                       p.rows, p.weights, p.pairs, p.experts, p.batch, route, place, list, count, p.bad);
    int code = plm::check_launch("pair lists");
    if (code != 0) return code;
    hipLaunchKernelGGL(pair_bases_kernel, dim3(1), dim3(64), 0, st, count, base, p.experts);
    if ((code = plm::check_launch("pair bases")) != 0) return code;
    for (int phase = 0; phase < 2; ++phase)
        for (int64_t g0 = 0; g0 < p.experts; g0 += kBatchGroups) {
            BatchRows b;
            b.ngroups = static_cast<int>(std::min<int64_t>(kBatchGroups, p.experts - g0));
            for (int g = 0; g < b.ngroups; ++g) {
                for (int i = 0; i < 2; ++i) {
                    b.w[i][g] = p.w[phase == 0 ? i : 2][g0 + g];
                    b.s[i][g] = p.s[phase == 0 ? i : 2][g0 + g];
                }
            }
            b.m = p.batch;
            b.groups.count = count + g0;
            b.groups.base = base + g0;
            if (phase == 0) {
                b.x = p.x;
                b.xb = p.xb;
                b.x_stride = p.hid;
                b.hhi = planes;
                b.hlo = planes + slots * p.inter;
                b.rows = p.inter;
                b.K = p.hid;
                b.scale_cols = p.gsc;
                b.waves = p.gate_waves;
                b.groups.list = list + g0 * p.batch;
                b.groups.list_ld = p.batch;
            } else {
                b.xhi = planes;
                b.xlo = planes + slots * p.inter;
                b.x_stride = p.inter;
                b.out = part;
                b.rows = p.hid;
                b.K = p.inter;
                b.scale_cols = p.dsc;
                b.waves = static_cast<int>(std::min<int64_t>(plm::ceil_div(p.inter, 128), kBatchDownWaves));
            }
            if ((code = fp8_batch_rows(b, st)) != 0) return code;
        }
    hipLaunchKernelGGL(pair_sum_kernel,
                       dim3(static_cast<unsigned>(p.batch), static_cast<unsigned>(plm::ceil_div(p.hid, 4 * kPairThreads))),
                       dim3(kPairThreads), 0, st, part, route, place, base, p.experts, p.batch, p.hid, p.out);
    return plm::check_launch("pair sum");
}
