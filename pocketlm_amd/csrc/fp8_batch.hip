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
// Measured on an MI355X against passes of 8 rows: 24576x1536 at 509 bf16 rows
// 787 -> 289 us, the 7168/2048 MLP at 256 fp32 rows 991 -> 251 us, 96 rows of
// top-8 over 256 experts of 7168/2048 27.2 -> 2.02 ms (5.3 TB/s: the weights
// of every chosen expert, read once).
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
};


// A workgroup owns 16 TA rows of each of its NWT weights; wave w of nw takes
// the K blocks w, w + nw, ... for all 16 TB activation rows of a pass.
template <int TA, int TB, int P, int NWT, bool SILU, int XM, int MAXW>
__global__ __launch_bounds__(64 * MAXW) void fp8_batch_kernel(const BatchArgs a) {
    constexpr int NT = NWT * TA;
    constexpr int PL = XM == kXPlanes ? 2 : 1;  // planes of the activations, with accumulators of their own
    constexpr bool XB = XM != kXF32;
    constexpr int XE = XB ? 2 : 4;
    extern __shared__ plm_f32x4 red[];  // [wave][tile][lane]
    const int nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int li = lane & 15, qd = lane >> 4;
    const int g = blockIdx.x / a.tiles;
    const int64_t row0 = static_cast<int64_t>(blockIdx.x - g * a.tiles) * 16 * TA;
    const int64_t count = a.count != nullptr ? a.count[g] : a.m;
    const int64_t obase = a.base != nullptr ? a.base[g] : g * a.m;

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
            const int64_t r = min(row0 + 16 * t + li, a.rows - 1);
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
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const bool in = !ragged || b * 128 + 64 * h + 16 * qd < K;
                        plm_bf16x8 a0[NT], a1[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            plm_u32x4 qv = q[slot][h][t];
                            if (ragged) qv = in ? qv : plm_u32x4{0, 0, 0, 0};
                            weights_to_bf16(SAN ? zero_nan_bytes(qv) : qv, a0[t], a1[t]);
                        }
#pragma unroll
                        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                            for (int pl = 0; pl < PL; ++pl) {
                                XPiece<XB> xv = x[slot][h][pl][tb];
                                if (ragged) {
#pragma unroll
                                    for (int i = 0; i < (XB ? 2 : 4); ++i)
                                        xv.v[i] = in ? xv.v[i] : plm_u32x4{0, 0, 0, 0};
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
            if (row >= a.rows || t >= count) continue;
            float v[NWT];
#pragma unroll
            for (int i = 0; i < NWT; ++i) {
                const int at = (((i * TA + ta) * TB + tb) * 64 + (r >> 2) * 16 + n) * 4 + (r & 3);
                float s = 0.0f;
                for (int w = 0; w < nw; ++w) s += rf[w * NT * TB * 256 + at];
                v[i] = s;
            }
            const int64_t o = (obase + t) * a.rows + row;
            if constexpr (SILU)
                store_hplanes(a.hhi, a.hlo, o, plm_silu_mul(v[0], v[1]));
            else
                a.out[o] = v[0];
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
    if (m <= 16)
        return xm == kXBf16 ? launch<2, 1, 2, 1, false, kXBf16, 8>(p, a, chunks(1), st)
                            : launch<2, 1, 2, 1, false, kXF32, 8>(p, a, chunks(1), st);
    if (m <= 32)
        return xm == kXBf16 ? launch<2, 2, 2, 1, false, kXBf16, 8>(p, a, chunks(2), st)
                            : launch<2, 2, 1, 1, false, kXF32, 8>(p, a, chunks(2), st);
    return xm == kXBf16 ? launch<2, 4, 1, 1, false, kXBf16, 8>(p, a, chunks(4), st)
                        : launch<2, 2, 1, 1, false, kXF32, 8>(p, a, chunks(2), st);
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
