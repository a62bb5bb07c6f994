// fp32 complex products on v_mfma_f32_16x16x4f32: operand lane (l16, g) supplies
// row / column l16 at k = g, the accumulator lane holds C[4 g + r][l16].
#pragma once

#include "common.h"

namespace qpam {

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Gauss accumulation of a complex product over k: t1 += ar br, t2 += ai bi,
// t3 += (ar + ai)(br + bi); then re = t1 - t2, im = t3 - t1 - t2.  Three real
// MFMAs per complex product instead of four.
struct Gauss {
    floatx4 t1, t2, t3;
};
__device__ __forceinline__ void gz(Gauss &x) {
    x.t1 = x.t2 = x.t3 = floatx4{0.f, 0.f, 0.f, 0.f};
}
__device__ __forceinline__ void gstep(Gauss &x, float ar, float ai, float br, float bi) {
    x.t1 = mfma4(ar, br, x.t1);
    x.t2 = mfma4(ai, bi, x.t2);
    x.t3 = mfma4(ar + ai, br + bi, x.t3);
}
__device__ __forceinline__ floatx4 gre(const Gauss &x) { return x.t1 - x.t2; }
__device__ __forceinline__ floatx4 gim(const Gauss &x) { return x.t3 - x.t1 - x.t2; }

// The same product with every real part summed on its own, re in one sum and im in
// another: four MFMAs, but no im = t3 - t1 - t2 from sums that each carry their own
// rounding (and an infinite part of an operand stays out of the other part).  conj:
// of neither operand, of a, or of b.
struct Plain {
    floatx4 re, im;
};
__device__ __forceinline__ void pz(Plain &x) { x.re = x.im = floatx4{0.f, 0.f, 0.f, 0.f}; }
__device__ __forceinline__ void pstep(Plain &x, float ar, float ai, float br, float bi) {
    x.re = mfma4(ar, br, x.re);
    x.im = mfma4(ar, bi, x.im);
    x.re = mfma4(ai, -bi, x.re);
    x.im = mfma4(ai, br, x.im);
}
__device__ __forceinline__ void pstep_ca(Plain &x, float ar, float ai, float br, float bi) {
    x.re = mfma4(ar, br, x.re);
    x.im = mfma4(ar, bi, x.im);
    x.re = mfma4(ai, bi, x.re);
    x.im = mfma4(ai, -br, x.im);
}
__device__ __forceinline__ void pstep_cb(Plain &x, float ar, float ai, float br, float bi) {
    x.re = mfma4(ar, br, x.re);
    x.im = mfma4(ar, -bi, x.im);
    x.re = mfma4(ai, bi, x.re);
    x.im = mfma4(ai, br, x.im);
}

// Interleaved complex LDS tiles: 64 rows of pitch CP.  One 8-byte read gives both
// parts of an operand down a column, two 16-byte reads four consecutive ones along
// a row; CP = 68 puts the four lane groups' rows 4 g + r of a column read on
// distinct banks.
constexpr int CP = 64 + 4;     // row pitch, complex elements
constexpr int TILE = 64 * CP;  // complex elements of a tile

// operand reads of a tile: four consecutive elements of a row from column k (16-byte
// aligned), or one element down a column
struct Four {
    float re[4], im[4];
};
__device__ __forceinline__ Four row4(const float2 *t, int row, int k) {
    const float4 a = *reinterpret_cast<const float4 *>(t + row * CP + k);
    const float4 b = *reinterpret_cast<const float4 *>(t + row * CP + k + 2);
    return Four{{a.x, a.z, b.x, b.z}, {a.y, a.w, b.y, b.w}};
}
__device__ __forceinline__ void put4(float2 *t, int row, int k, const floatx4 &re, const floatx4 &im) {
    *reinterpret_cast<float4 *>(t + row * CP + k) = make_float4(re[0], im[0], re[1], im[1]);
    *reinterpret_cast<float4 *>(t + row * CP + k + 2) = make_float4(re[2], im[2], re[3], im[3]);
}

}  // namespace qpam
