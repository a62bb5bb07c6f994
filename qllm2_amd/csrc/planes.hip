// Split-real [..., d, 2] tensors to and from the planar operands of the scan
// and delta kernels: up to QPAM_PLANES_MAX tensors in one launch, each with
// its own strides and element types, planes zero-padded to the kernels' head
// dim on the way in.  A pure copy, bound by HBM.  A thread moves four complex
// elements (16-byte accesses on both sides in fp32), neighbouring threads the
// neighbouring groups of a row, so both sides are read and written in whole
// cache lines.  fp32 calls of head dim 64 pass here with q, k, v and the state only (their
// y and gradients leave the kernels as split-real rows); the others also with y, dy and
// the gradients.  At B=8, H=12, T=2048, d=64 fp32 (100 MB a tensor) splitting q, k, v moves
// 604 MB in 91 us = 6.6 TB/s; a step that copies all eight tensors moves 1.6 GB in
// 265 us, where the slices, zero fills, adds and stacks of the library took 870 us.
#include "common.h"

namespace qpam {
namespace {

constexpr int PL_THREADS = 256;

template <typename T>
__device__ __forceinline__ void il_load(const void *p, int64_t o, int n, bool vec, float (&re)[4], float (&im)[4]);
template <>
__device__ __forceinline__ void il_load<float>(const void *p, int64_t o, int n, bool vec, float (&re)[4], float (&im)[4]) {
    const float *s = static_cast<const float *>(p) + o;
    if (vec) {
        const float4 a = reinterpret_cast<const float4 *>(s)[0], b = reinterpret_cast<const float4 *>(s)[1];
        re[0] = a.x, im[0] = a.y, re[1] = a.z, im[1] = a.w, re[2] = b.x, im[2] = b.y, re[3] = b.z, im[3] = b.w;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) re[e] = e < n ? s[2 * e] : 0.f, im[e] = e < n ? s[2 * e + 1] : 0.f;
    }
}
template <>
__device__ __forceinline__ void il_load<unsigned short>(const void *p, int64_t o, int n, bool vec, float (&re)[4],
                                                        float (&im)[4]) {
    const unsigned short *s = static_cast<const unsigned short *>(p) + o;
    if (vec) {
        const ushortx8 a = *reinterpret_cast<const ushortx8 *>(s);
#pragma unroll
        for (int e = 0; e < 4; ++e) re[e] = bf16_to_f32(a[2 * e]), im[e] = bf16_to_f32(a[2 * e + 1]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            re[e] = e < n ? bf16_to_f32(s[2 * e]) : 0.f, im[e] = e < n ? bf16_to_f32(s[2 * e + 1]) : 0.f;
    }
}

template <typename T>
__device__ __forceinline__ void il_store(void *p, int64_t o, int n, bool vec, const float (&re)[4], const float (&im)[4]);
template <>
__device__ __forceinline__ void il_store<float>(void *p, int64_t o, int n, bool vec, const float (&re)[4],
                                                const float (&im)[4]) {
    float *s = static_cast<float *>(p) + o;
    if (vec) {
        reinterpret_cast<float4 *>(s)[0] = make_float4(re[0], im[0], re[1], im[1]);
        reinterpret_cast<float4 *>(s)[1] = make_float4(re[2], im[2], re[3], im[3]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < n) s[2 * e] = re[e], s[2 * e + 1] = im[e];
    }
}
template <>
__device__ __forceinline__ void il_store<unsigned short>(void *p, int64_t o, int n, bool vec, const float (&re)[4],
                                                         const float (&im)[4]) {
    unsigned short *s = static_cast<unsigned short *>(p) + o;
    const uintx4 u = {pack_bf16x2(re[0], im[0]), pack_bf16x2(re[1], im[1]), pack_bf16x2(re[2], im[2]),
                      pack_bf16x2(re[3], im[3])};
    if (vec) {
        *reinterpret_cast<uintx4 *>(s) = u;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < n) s[2 * e] = (unsigned short)u[e], s[2 * e + 1] = (unsigned short)(u[e] >> 16);
    }
}

template <typename T>
__device__ __forceinline__ void pl_load(const void *p, int64_t o, int n, bool vec, float (&x)[4]) {
    const T *s = static_cast<const T *>(p) + o;
    if (vec) {
        if constexpr (sizeof(T) == 4) {
            const float4 a = *reinterpret_cast<const float4 *>(s);
            x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w;
        } else {
            const ushortx4 a = *reinterpret_cast<const ushortx4 *>(s);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = bf16_to_f32(a[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = e < n ? Elem<T>::load(s + e) : 0.f;
    }
}
// planes are written in whole groups of four: their width is a multiple of 4
template <typename T>
__device__ __forceinline__ void pl_store(void *p, int64_t o, const float (&x)[4]) {
    T *s = static_cast<T *>(p) + o;
    if constexpr (sizeof(T) == 4) {
        *reinterpret_cast<float4 *>(s) = make_float4(x[0], x[1], x[2], x[3]);
    } else {
        typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
        *reinterpret_cast<uintx2 *>(s) = uintx2{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
    }
}

struct PlanesParams {
    qpam_planes_item it[QPAM_PLANES_MAX];
    int32_t vec[QPAM_PLANES_MAX];
};

// item blockIdx.y; thread = one group of four columns of one plane row (i0, i1, i2)
template <bool MERGE>
__global__ void __launch_bounds__(PL_THREADS) planes_kernel(PlanesParams p) {
    const qpam_planes_item it = p.it[blockIdx.y];
    const bool vec = p.vec[blockIdx.y];
    const unsigned groups = (unsigned)((MERGE ? it.d + 3 : it.dp) / 4);
    const unsigned rows = MERGE ? it.n2_il : it.n2;
    const unsigned total = (unsigned)it.n0 * it.n1 * rows * groups;
    unsigned e = blockIdx.x * PL_THREADS + threadIdx.x;
    if (e >= total) return;
    const unsigned g = e % groups;
    e /= groups;
    const unsigned i2 = e % rows;
    e /= rows;
    const unsigned i1 = e % (unsigned)it.n1, i0 = e / (unsigned)it.n1;
    const int64_t lo = i0 * it.l0 + i1 * it.l1 + i2 * it.l2 + 8 * (int64_t)g;
    const int64_t po = i0 * it.p0 + i1 * it.p1 + i2 * it.p2 + 4 * (int64_t)g;
    const int n = (int)it.d - 4 * (int)g;
    float re[4] = {0.f, 0.f, 0.f, 0.f}, im[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (MERGE) {
        if (it.pl_dtype == QPAM_BF16) {
            pl_load<unsigned short>(it.re, po, n, vec, re), pl_load<unsigned short>(it.im, po, n, vec, im);
        } else {
            pl_load<float>(it.re, po, n, vec, re), pl_load<float>(it.im, po, n, vec, im);
        }
        if (it.il_dtype == QPAM_BF16) il_store<unsigned short>(it.il, lo, n, vec, re, im);
        else il_store<float>(it.il, lo, n, vec, re, im);
    } else {
        if (n > 0 && i2 < (unsigned)it.n2_il) {
            if (it.il_dtype == QPAM_BF16) il_load<unsigned short>(it.il, lo, n, vec, re, im);
            else il_load<float>(it.il, lo, n, vec, re, im);
        }
        if (it.pl_dtype == QPAM_BF16) pl_store<unsigned short>(it.re, po, re), pl_store<unsigned short>(it.im, po, im);
        else pl_store<float>(it.re, po, re), pl_store<float>(it.im, po, im);
    }
}

bool mult(int64_t a, int64_t b, int64_t c, int64_t m) { return a % m == 0 && b % m == 0 && c % m == 0; }

}  // namespace
}  // namespace qpam

using namespace qpam;

extern "C" int qpam_planes(const qpam_planes_args *a, void *stream) {
    QPAM_REQUIRE(a != nullptr, "qpam_planes: null args");
    QPAM_REQUIRE(a->count >= 1 && a->count <= QPAM_PLANES_MAX, "qpam_planes: 1 to %d tensors", QPAM_PLANES_MAX);
    QPAM_REQUIRE(a->merge == 0 || a->merge == 1, "qpam_planes: merge must be 0 or 1");
    PlanesParams p;
    int64_t most = 0;
    for (int i = 0; i < a->count; ++i) {
        const qpam_planes_item &it = a->item[i];
        QPAM_REQUIRE(it.n0 >= 0 && it.n1 >= 0 && it.n2 >= it.n2_il && it.n2_il >= 0 && it.d >= 1 && it.dp >= it.d &&
                         it.dp % 4 == 0,
                     "qpam_planes: sizes of tensor %d", i);
        QPAM_REQUIRE((it.il_dtype == QPAM_F32 || it.il_dtype == QPAM_BF16) &&
                         (it.pl_dtype == QPAM_F32 || it.pl_dtype == QPAM_BF16),
                     "qpam_planes: dtypes must be QPAM_F32 or QPAM_BF16");
        const int64_t rows = a->merge ? it.n2_il : it.n2, groups = (a->merge ? it.d + 3 : it.dp) / 4;
        const int64_t total = (int64_t)it.n0 * it.n1 * rows * groups;
        QPAM_REQUIRE(total < (1ll << 31), "qpam_planes: tensor %d too large", i);
        const int64_t pb = it.pl_dtype == QPAM_BF16 ? 8 : 16;
        const bool pl_ok = mult(it.p0, it.p1, it.p2, 4) && ((uintptr_t)it.re | (uintptr_t)it.im) % pb == 0;
        QPAM_REQUIRE(total == 0 || (it.il && it.re && it.im), "qpam_planes: null tensor %d", i);
        QPAM_REQUIRE(a->merge || pl_ok, "qpam_planes: planes of tensor %d must be 16-byte aligned rows", i);
        const int64_t lm = it.il_dtype == QPAM_BF16 ? 8 : 4;
        p.it[i] = it;
        p.vec[i] = pl_ok && it.d % 4 == 0 && mult(it.l0, it.l1, it.l2, lm) && (uintptr_t)it.il % 16 == 0;
        most = total > most ? total : most;
    }
    if (most == 0) return QPAM_OK;
    const dim3 grid((unsigned)((most + PL_THREADS - 1) / PL_THREADS), (unsigned)a->count);
    if (a->merge) hipLaunchKernelGGL(planes_kernel<true>, grid, dim3(PL_THREADS), 0, (hipStream_t)stream, p);
    else hipLaunchKernelGGL(planes_kernel<false>, grid, dim3(PL_THREADS), 0, (hipStream_t)stream, p);
    return launch_status("planes_kernel");
}
