// Device helpers of the FP8 e4m3 block-scaled kernels on the matrix cores:
// vector loads, e4m3 -> bf16, fp32 -> bf16 hi + lo, and the register
// pipeline of a wave (fp8_gemv.hip, fp8_batch.hip).
#pragma once

#include "common.h"

namespace plm_fp8 {

typedef __bf16 plm_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 plm_bf16x2 __attribute__((ext_vector_type(2)));
typedef float plm_f32x4 __attribute__((ext_vector_type(4)));

// Weight bytes are read once per call: nontemporal loads keep them from
// displacing the activations and scales in the caches.
__device__ __forceinline__ plm_u32x4 wload16(const void* p) {
    return __builtin_nontemporal_load((const __attribute__((address_space(1))) plm_u32x4*)(p));
}

__device__ __forceinline__ plm_u32x4 xload16(const void* p) {
    return *(const __attribute__((address_space(1))) plm_u32x4*)(p);
}

template <bool HI>
__device__ __forceinline__ uint32_t e4m3_pair_to_bf16(uint32_t v) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, HI));
}

// 16 e4m3 bytes -> the two A operands (bytes 0-7, 8-15)
__device__ __forceinline__ void weights_to_bf16(const plm_u32x4 q, plm_bf16x8& a0, plm_bf16x8& a1) {
    const plm_u32x4 t0 = {e4m3_pair_to_bf16<false>(q.x), e4m3_pair_to_bf16<true>(q.x),
                          e4m3_pair_to_bf16<false>(q.y), e4m3_pair_to_bf16<true>(q.y)};
    const plm_u32x4 t1 = {e4m3_pair_to_bf16<false>(q.z), e4m3_pair_to_bf16<true>(q.z),
                          e4m3_pair_to_bf16<false>(q.w), e4m3_pair_to_bf16<true>(q.w)};
    a0 = __builtin_bit_cast(plm_bf16x8, t0);
    a1 = __builtin_bit_cast(plm_bf16x8, t1);
}

// NaN bytes (0x7F, 0xFF) -> 0
__device__ __forceinline__ plm_u32x4 zero_nan_bytes(plm_u32x4 q) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t w = q[k];
        const uint32_t nan = ((w & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u;  // 0x80 where the low 7 bits are all 1
        q[k] = w & ~((nan >> 7) * 0xFFu);
    }
    return q;
}

// hi / lo bf16 halves of one fp32 value.  EXACT: infinities and NaNs go to hi
// whole (a quiet NaN for every NaN) with lo = 0.
template <bool EXACT>
__device__ __forceinline__ void split_f32(uint32_t x, uint32_t& hi, uint32_t& lo) {
    hi = x >> 16;
    const float rem = __uint_as_float(x) - __uint_as_float(x & 0xFFFF0000u);
    lo = __builtin_bit_cast(uint16_t, static_cast<__bf16>(rem));
    if constexpr (EXACT) {
        if ((x & 0x7F800000u) == 0x7F800000u) {
            hi = (x & 0x007FFFFFu) != 0 ? 0x7FC0u : hi;
            lo = 0;
        }
    }
}

// 8 fp32 activations (two loads) -> hi and lo B operands
template <bool EXACT>
__device__ __forceinline__ void split8(const plm_u32x4 v0, const plm_u32x4 v1, plm_bf16x8& hi, plm_bf16x8& lo) {
    const uint32_t x[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
    plm_u32x4 h, l;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        if constexpr (EXACT) {
            uint32_t h0, l0, h1, l1;
            split_f32<true>(x[2 * p], h0, l0);
            split_f32<true>(x[2 * p + 1], h1, l1);
            h[p] = h0 | (h1 << 16);
            l[p] = l0 | (l1 << 16);
        } else {
            h[p] = __builtin_amdgcn_perm(x[2 * p + 1], x[2 * p], 0x07060302u);
            const float r0 = __uint_as_float(x[2 * p]) - __uint_as_float(x[2 * p] & 0xFFFF0000u);
            const float r1 = __uint_as_float(x[2 * p + 1]) - __uint_as_float(x[2 * p + 1] & 0xFFFF0000u);
            const plm_float2 rr = {r0, r1};
            l[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rr, plm_bf16x2));
        }
    }
    hi = __builtin_bit_cast(plm_bf16x8, h);
    lo = __builtin_bit_cast(plm_bf16x8, l);
}

__device__ __forceinline__ plm_f32x4 mfma_bf16(plm_bf16x8 a, plm_bf16x8 b, plm_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The activations of one block for the lane's B column: two bf16 loads, or
// four fp32 loads (split into hi and lo later).
template <bool XB>
struct XPiece {
    plm_u32x4 v[XB ? 2 : 4];
};

template <bool XB>
__device__ __forceinline__ XPiece<XB> load_xpiece(const void* p, bool live) {
    XPiece<XB> r;
    const char* c = static_cast<const char*>(p);
#pragma unroll
    for (int k = 0; k < (XB ? 2 : 4); ++k) r.v[k] = live ? xload16(c + 16 * k) : plm_u32x4{0, 0, 0, 0};
    return r;
}

template <bool XB, bool SAN>
struct BOperands {
    plm_bf16x8 h0, h1, l0, l1;
    BOperands() = default;
    __device__ __forceinline__ explicit BOperands(const XPiece<XB>& x) {
        if constexpr (XB) {
            h0 = __builtin_bit_cast(plm_bf16x8, x.v[0]);
            h1 = __builtin_bit_cast(plm_bf16x8, x.v[1]);
        } else {
            split8<SAN>(x.v[0], x.v[1], h0, l0);
            split8<SAN>(x.v[2], x.v[3], h1, l1);
        }
    }
};

// The SiLU intermediate silu(gate) * up as the down phase reads it: bf16
// hi / lo planes (exact for infinities and NaNs).
__device__ __forceinline__ void store_hplanes(uint16_t* hi, uint16_t* lo, int64_t o, float v) {
    uint32_t h, l;
    split_f32<true>(__float_as_uint(v), h, l);
    hi[o] = static_cast<uint16_t>(h);
    lo[o] = static_cast<uint16_t>(l);
}

__device__ __forceinline__ float lane_value(float v, int k) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}

// Runs nk steps through P register slots, pipelined: P steps are in
// flight and step k + P is issued into the slot step k leaves; the steps
// beyond a multiple of P run first, unpipelined.
template <int P, class Issue, class Compute>
__device__ __forceinline__ void run_pipelined(int nk, Issue& issue, Compute& compute) {
    const int r = nk % P;
    for (int k = 0; k < r; ++k) {
        issue(0, k);
        compute(0, k);
    }
    if (nk > r) {
#pragma unroll
        for (int u = 0; u < P; ++u) issue(u, r + u);
        for (int k0 = r; k0 + P < nk; k0 += P) {
#pragma unroll
            for (int u = 0; u < P; ++u) {
                compute(u, k0 + u);
                issue(u, k0 + u + P);
            }
        }
#pragma unroll
        for (int u = 0; u < P; ++u) compute(u, nk - P + u);
    }
}

}  // namespace plm_fp8
