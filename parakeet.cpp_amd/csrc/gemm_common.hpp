// Device helpers shared by the GEMM sources: slab-major weight addressing, the
// XCD-aware tile order and the element epilogues.
#pragma once
#include "gemm.hpp"

namespace pkx {

// Rows of each 64-wide K slab block of a slab-major (q8_0 / q4_K) weight (views
// into a larger allocation keep the allocation's row count).
__device__ __forceinline__ int slab_rows(const GemmParams& p) { return p.ldw > 0 ? p.ldw : p.N; }

// Exact int8 -> f16 for 4 packed bytes: byte b (two's complement) becomes the
// f16 with bit pattern 0x6400 | (b ^ 0x80) = 1024 + (b + 128); subtracting
// 1152 leaves b exactly.  Then one correctly rounded f16 multiply by d.
__device__ __forceinline__ void i8x4_to_f16(uint32_t w, half2v d2, half2v& lo, half2v& hi) {
    const uint32_t u = w ^ 0x80808080u;
    const uint32_t a = __builtin_amdgcn_perm(0x64646464u, u, 0x07010700u) ;  // [0x64,b1,0x64,b0]
    const uint32_t b = __builtin_amdgcn_perm(0x64646464u, u, 0x07030702u);   // [0x64,b3,0x64,b2]
    const half2v bias = {(f16)1152.0f, (f16)1152.0f};
    lo = (__builtin_bit_cast(half2v, a) - bias) * d2;
    hi = (__builtin_bit_cast(half2v, b) - bias) * d2;
}

// Four 4-bit weights (nibble `hi` of each byte of w) to f16, w = s*q - m with
// nm2 = -m: the nibble is placed in an f16 mantissa so that the half reads
// 1024 + q (low nibble, exponent byte 0x64) or 64 + q (high nibble in mantissa
// bits 4..7, exponent byte 0x54); subtracting 1024 or 64 is exact, then one
// rounding in the fma.
__device__ __forceinline__ void nib4_to_f16(uint32_t w, int hi, half2v s2, half2v nm2, half2v& lo, half2v& up) {
    const uint32_t e = hi ? 0x54545454u : 0x64646464u;
    const uint32_t mask = hi ? 0xFFF0FFF0u : 0xFF0FFF0Fu;
    const f16 off = hi ? (f16)64.0f : (f16)1024.0f;
    const half2v off2 = {off, off};
    const uint32_t a = __builtin_amdgcn_perm(e, w, 0x07010700u) & mask;  // bytes 0, 1
    const uint32_t b = __builtin_amdgcn_perm(e, w, 0x07030702u) & mask;  // bytes 2, 3
    lo = (__builtin_bit_cast(half2v, a) - off2) * s2 + nm2;
    up = (__builtin_bit_cast(half2v, b) - off2) * s2 + nm2;
}

// 2-D XCD blocking: the nbm x nbn tile grid is cut into gm row bands x gn
// column bands (gm * gn = 8), one rectangle per XCD, so an XCD's L2 sees only
// its band of A rows and its band of weight columns (gn*|A| + gm*|W| bytes
// over the chip instead of 8*|A| or 8*|W|).  xcd_tile gives each XCD a
// contiguous range of positions; positions enumerate the rectangles in order,
// each rectangle M-fastest, so the map is a bijection for any grid size.
// gm and gn are powers of two, so the band edges i * nbm / gm are shifts; the
// one division left is the split of k inside its rectangle.  (With a division
// for every band edge this ran ~3k cycles at the start of every launch, all
// of it before the first load: 32-bit division by a runtime value is a
// ~40-instruction scalar / vector round trip on this hardware.)
__device__ __forceinline__ void xcd_rect(int k, int nbm, int nbn, int gm, int& bm, int& bn) {
    const int lgm = __builtin_ctz(gm), lgn = 3 - lgm;
    for (int i = 0; i < gm; ++i) {
        const int r0 = (i * nbm) >> lgm, r1 = ((i + 1) * nbm) >> lgm;
        for (int j = 0; j < (1 << lgn); ++j) {
            const int c0 = (j * nbn) >> lgn, c1 = ((j + 1) * nbn) >> lgn;
            const int h = r1 - r0, sz = h * (c1 - c0);
            if (k < sz) {   // sz > 0, so h > 0
                const int q = (int)((unsigned)k / (unsigned)h);
                bm = r0 + (k - q * h);
                bn = c0 + q;
                return;
            }
            k -= sz;
        }
    }
    bm = bn = 0;   // unreachable: the rectangles cover the grid
}
__device__ __forceinline__ void xcd_tile_2d(int bid, int nbm, int nbn, int gm, int& bm, int& bn) {
    xcd_rect(xcd_tile(bid, nbm * nbn), nbm, nbn, gm, bm, bn);
}

// ---------------------------------------------------------------------------
// Epilogue for one accumulator element (everything except GLU).
// ---------------------------------------------------------------------------
template <int EPI, typename ActT>
__device__ __forceinline__ void epi_one(const GemmParams& p, int m, int n, float acc) {
    float v = acc + (p.bias ? p.bias[n] : 0.0f);
    if constexpr (EPI == EPI_STORE) {
        ((ActT*)p.Y)[(int64_t)m * p.ldy + n] = to_act<ActT>(v * p.alpha);
    } else if constexpr (EPI == EPI_STORE_F32) {
        ((float*)p.Y)[(int64_t)m * p.ldy + n] = v * p.alpha;
    } else if constexpr (EPI == EPI_SILU) {
        ((ActT*)p.Y)[(int64_t)m * p.ldy + n] = to_act<ActT>(silu_dev(v));
    } else if constexpr (EPI == EPI_RESID) {
        float* r = (float*)p.Y + (int64_t)m * p.ldy + n;
        *r = *r + v * p.alpha;
    } else if constexpr (EPI == EPI_RELU) {
        ((ActT*)p.Y)[(int64_t)m * p.ldy + n] = to_act<ActT>(v > 0.f ? v : 0.f);
    } else if constexpr (EPI == EPI_RELU_TR) {
        // rows are pixels (b, t, f), f fastest; store [b][t][c][f] (channel-major flatten)
        const int F = p.trF;
        const int bt = m / F, f = m - bt * F;
        const int t = bt % p.T, b = bt / p.T;
        float o = v > 0.f ? v : 0.f;
        if (p.valid && t >= p.valid[b]) o = 0.f;
        ((ActT*)p.Y)[((int64_t)bt * p.N + n) * F + f] = to_act<ActT>(o);
    } else if constexpr (EPI == EPI_RELU2_F32) {
        float o = v + (p.bias2 ? p.bias2[n] : 0.0f);
        ((float*)p.Y)[(int64_t)m * p.ldy + n] = o > 0.f ? o : 0.f;
    }
}

// gemm_rows.hip: one f16 product of few rows on K-split tiles where that is the
// faster kernel; false (nothing launched) where it is not.
bool launch_gemm_rows(int wtype, int epi, const GemmParams& p, hipStream_t s);

// gemm_f32.hip: one f32 product with f32 weights on K-split tiles where that is
// the faster kernel; false (nothing launched) where it is not.
bool launch_gemm_f32_ks(int epi, const GemmParams& p, hipStream_t s);

}  // namespace pkx
