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

}  // namespace qpam
