// E1 per-channel decay, forward and backward of the chunked form for head dims
// up to 64 (V11PAMLayer._forward_chunked_perchannel, v11/model.py:421-489).
// With L the clamped log-decay prefix of a chunk per key channel,
//   Qf = q e^{L} q_scale, Kf = k e^{-L}, W = k e^{L_last - L} = Kf E, E_j = e^{L_last[j]},
//   P = tril(Qf Kf^H),  y = P V + Qf S^T,  S <- E S + V^T conj(W)   (E scales column j),
// each chunk is a handful of 64 x 64 complex products on fp32 MFMA (gauss.h)
// whose operands are folded on the way into LDS, so nothing but the chunk states
// passes through HBM between the launches:
//   forward:  pc_state (increments V^T conj(W)) -> qpam_pc_scan -> pc_output
//   backward: pc_state (increments dY^T conj(Qf)) -> qpam_pc_scan in reverse -> pc_grad
// At B=8, H=12, T=2048, d=64, chunk 64 (fp32) a training step takes 1.04 ms (was
// 2.64 ms: twelve batched library products whose operands and results each crossed
// HBM, 1.36 ms, the fold kernels, 0.41 ms, and conjugations, transposes, masks and
// sums).  The kernels are bound by each block's load, product and store phases
// following one another at one to three blocks per CU, more than by the matrix cores.
// Precision: every real part of a product is summed on its own (gauss.h, Plain).  With
// three MFMAs per product, e^{L} and e^{-L} by __expf, and W formed as Kf E, the step
// took 1.01 ms, but the imaginary planes of y, s, dk and dv were 1.03-1.31 times as far
// from 64 bits as the library products' (now 0.80-1.02, within chance), and prefixes
// near -30 cost dk and dv 1.12-1.14 in both planes: expf where both e^{L} and e^{-L}
// enter a result, W by its own exponential.
//
// Tiles are staged by lane = column, so a wave's access to a row is one 512-byte run.
#include "gauss.h"

namespace qpam {
namespace {

constexpr int CH = 64;                   // rows of a kernel chunk (steps past the chunk's are zero)
// A grid holds at most 2^32 - 1 threads along an axis (one past it wraps without an
// error): chunks beyond 2^20 go on along y, up to 65535 rows of them.
constexpr int64_t GRID_X = 1 << 20;
constexpr float GAMMA_FLOOR = 1e-6f;     // gamma.clamp_min(1e-6), v11/model.py:436
constexpr float CUM_FLOOR = -30.f;       // cumsum.clamp(min=-30), v11/model.py:438

// Accesses take a wave-uniform row offset and a 32-bit lane offset (elements), so
// an address costs scalar registers and one lane offset shared by every row.
// An element is loaded as it lies in memory (a bf16 pair in .x) and widened where it
// is used, so the type is branched on once per tensor and no load waits for another.
__device__ __forceinline__ float2 widen(float2 x, int dt) {
    const unsigned u = __float_as_uint(x.x);
    return dt == QPAM_BF16 ? make_float2(__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u)) : x;
}
__device__ __forceinline__ float widen(float x, int dt) {
    return dt == QPAM_BF16 ? __uint_as_float(__float_as_uint(x) << 16) : x;
}
__device__ __forceinline__ void st_c(void *p, int64_t row, unsigned lane, float2 v, int dt) {
    if (dt == QPAM_BF16)
        *reinterpret_cast<unsigned *>(static_cast<unsigned short *>(p) + row + lane) = pack_bf16x2(v.x, v.y);
    else *reinterpret_cast<float2 *>(static_cast<float *>(p) + row + lane) = v;
}
// One chunk of one chain: lane j of wave grp owns channel j and steps
// ROWS grp .. ROWS grp + ROWS - 1.
template <int ROWS>
struct Pos {
    int64_t cc;  // chain * n + c
    int j, jc, grp, b, h, t0, valid;  // jc: j clamped into the channels
    bool jv;
    // blocks past the last chunk (in the grid's last row of several) have nothing to do
    __device__ __forceinline__ static bool past(const qpam_pc_args &a, int n) {
        return (int64_t)blockIdx.y * GRID_X + blockIdx.x >= a.B * a.H * n;
    }
    __device__ __forceinline__ Pos(const qpam_pc_args &a, int n) {
        cc = (int64_t)blockIdx.y * GRID_X + blockIdx.x;
        j = threadIdx.x & 63;
        grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar branches and row offsets
        const int c = (int)(cc % n);
        const int chain = (int)(cc / n);
        b = chain / (int)a.H;
        h = chain % (int)a.H;
        t0 = c * a.chunk;
        valid = (int)min((int64_t)a.chunk, a.T - t0);
        jv = j < a.d;
        jc = jv ? j : (int)a.d - 1;
    }
    __device__ __forceinline__ int row(int r) const { return ROWS * grp + r; }
    __device__ __forceinline__ bool ok(int r) const { return jv && row(r) < valid; }
    // element offset of the chunk's first step (wave-uniform)
    __device__ __forceinline__ int64_t at(int64_t sb, int64_t sh, int64_t st) const {
        return b * sb + h * sh + (int64_t)t0 * st;
    }
    // row r clamped into the chunk
    __device__ __forceinline__ int crow(int r) const { return min(row(r), valid - 1); }
};

// The lane's elements of its steps.  Rows past the chunk re-read its last step and
// channels past d the last channel: no load is conditional, so all are in flight
// together; keep() drops them where they are used.
template <int ROWS>
__device__ __forceinline__ void load_rows(float2 (&x)[ROWS], const Pos<ROWS> &p, const void *src, int64_t o, int64_t st,
                                          int dt) {
    const unsigned lane = 2u * p.jc;
    if (dt == QPAM_BF16) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
            x[r].x = *reinterpret_cast<const float *>(static_cast<const unsigned short *>(src) + o + p.crow(r) * st + lane);
    } else {
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
            x[r] = *reinterpret_cast<const float2 *>(static_cast<const float *>(src) + o + p.crow(r) * st + lane);
    }
}
template <int ROWS>
__device__ __forceinline__ void load_gamma(float (&x)[ROWS], const Pos<ROWS> &p, const qpam_pc_args &a) {
    const int64_t o = p.at(a.g_sb, a.g_sh, a.g_st);
    const unsigned lane = p.jc;
    if (a.g_dtype == QPAM_BF16) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
            x[r] = __uint_as_float((static_cast<const unsigned short *>(a.gamma) + o + p.crow(r) * a.g_st)[lane]);
    } else {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) x[r] = (static_cast<const float *>(a.gamma) + o + p.crow(r) * a.g_st)[lane];
    }
}
// rows i of the lane's column of a [d][d][2] matrix, with the same clamping
template <int ROWS>
__device__ __forceinline__ void load_state(float2 (&x)[ROWS], const Pos<ROWS> &p, const float *src, int64_t d) {
    const unsigned lane = 2u * p.jc;
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
        x[r] = *reinterpret_cast<const float2 *>(src + 2 * min((int64_t)p.row(r), d - 1) * d + lane);
}
__device__ __forceinline__ float2 keep(bool ok, float2 x, float f = 1.f) {
    return make_float2(ok ? x.x * f : 0.f, ok ? x.y * f : 0.f);
}

// gamma of the lane's steps (1 outside the sequence) -> unclamped inclusive prefixes
// cs of log max(gamma, floor) over the chunk (group totals through LDS, added in
// group order); returns the clamped L_last.  Two barriers.
template <int ROWS>
__device__ __forceinline__ float prefix(const Pos<ROWS> &p, const float (&gam)[ROWS], int dt, float (&cs)[ROWS],
                                        float *sTot, float *sLast) {
    float run = 0.f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        run += p.ok(r) ? logf(fmaxf(widen(gam[r], dt), GAMMA_FLOOR)) : 0.f;
        cs[r] = run;
    }
    sTot[p.grp * CH + p.j] = run;
    __syncthreads();
    float off = 0.f;
    for (int g = 0; g < p.grp; ++g) off += sTot[g * CH + p.j];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) cs[r] += off;
    // the prefix is constant from the chunk's last step on, so the last group's
    // last entry is the prefix at step valid - 1
    if (p.grp == CH / ROWS - 1) sLast[p.j] = fmaxf(cs[ROWS - 1], CUM_FLOOR);
    __syncthreads();
    return sLast[p.j];
}

// ------------------------------------------------------------- pc_state --
// Chunk increment X[i][j] = sum_t A[t][i] conj(B[t][j]): A = V, B = W (and the
// chunk's column decays E) in the forward, A = dY, B = Qf in the backward.  A block
// of 4 waves per (chain, chunk), wave w rows 16 w.. of X.  HBM-bound: reads two
// tensors and gamma, writes the increments.  The rows pass through LDS in two
// halves (36 KB): three blocks per CU, whose loads and products overlap (104 us =
// 3.4 TB/s at the shape above; 92 us with three MFMAs per product).
constexpr int ST_THREADS = 256, ST_ROWS = CH * 64 / ST_THREADS, ST_HALF = CH / 2;
constexpr size_t ST_SMEM = 2 * ST_HALF * CP * sizeof(float2) + (4 + 1) * CH * sizeof(float);

template <int DT, bool BWD>
__global__ void __launch_bounds__(ST_THREADS, 3) pc_state_kernel(qpam_pc_args a, int n) {
    extern __shared__ __align__(16) float2 smem[];
    float2 *sA = smem, *sB = sA + ST_HALF * CP;
    float *sTot = reinterpret_cast<float *>(sB + ST_HALF * CP), *sLast = sTot + 4 * CH;
    if (Pos<ST_ROWS>::past(a, n)) return;
    const Pos<ST_ROWS> p(a, n);
    float2 xa[ST_ROWS], xb[ST_ROWS];
    float gam[ST_ROWS], cs[ST_ROWS];
    load_gamma<ST_ROWS>(gam, p, a);
    if constexpr (BWD) {
        const int64_t so = (int64_t)a.T * a.d * 2;  // dy is contiguous [B,H,T,d,2]
        load_rows<ST_ROWS>(xb, p, a.q, p.at(a.q_sb, a.q_sh, a.q_st), a.q_st, a.dtype);
        load_rows<ST_ROWS>(xa, p, a.dy, p.at(a.H * so, so, 2 * a.d), 2 * a.d, a.dtype);
    } else {
        load_rows<ST_ROWS>(xb, p, a.k, p.at(a.k_sb, a.k_sh, a.k_st), a.k_st, a.dtype);
        load_rows<ST_ROWS>(xa, p, a.v, p.at(a.v_sb, a.v_sh, a.v_st), a.v_st, a.v_dtype);
    }
    const float Llast = prefix<ST_ROWS>(p, gam, a.g_dtype, cs, sTot, sLast);
    if (!BWD && p.grp == 0 && p.jv) a.atot[p.cc * a.d + p.j] = __expf(Llast);
    const int w = p.grp, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    Plain x[DT];
#pragma unroll
    for (int jt = 0; jt < DT; ++jt) pz(x[jt]);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (ST_HALF * half >= p.valid) break;  // rows past the chunk are zero
        if (half) __syncthreads();
        if (p.grp / 2 == half) {
#pragma unroll
            for (int r = 0; r < ST_ROWS; ++r) {
                const float L = fmaxf(cs[r], CUM_FLOOR);
                const float f = BWD ? __expf(L) * a.q_scale : __expf(Llast - L);
                const int o = (p.row(r) - ST_HALF * half) * CP + p.j;
                sA[o] = keep(p.ok(r), widen(xa[r], BWD ? a.dtype : a.v_dtype));
                sB[o] = keep(p.ok(r), widen(xb[r], a.dtype), f);
            }
        }
        __syncthreads();
        if (w < DT) {
#pragma unroll
            for (int ks = 0; ks < ST_HALF / 4; ++ks) {
                const int t = 4 * ks + g;
                const float2 u = sA[t * CP + 16 * w + l16];
#pragma unroll
                for (int jt = 0; jt < DT; ++jt) {
                    const float2 v = sB[t * CP + 16 * jt + l16];
                    pstep_cb(x[jt], u.x, u.y, v.x, v.y);
                }
            }
        }
    }
    if (w >= DT) return;
    float *dst = a.x + p.cc * a.d * a.d * 2;
#pragma unroll
    for (int jt = 0; jt < DT; ++jt) {
        const floatx4 re = x[jt].re, im = x[jt].im;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * w + 4 * g + r, j = 16 * jt + l16;
            if (i < a.d && j < a.d) st_c(dst, 0, 2u * ((unsigned)i * (unsigned)a.d + j), make_float2(re[r], im[r]), QPAM_F32);
        }
    }
}

// ------------------------------------------------------------ pc_output --
// y = P V + Qf S^T of one chunk: a block of 4 waves, wave w the query rows 16 w..;
// the score is formed transposed (its accumulator is the next product's operand)
// and one LDS tile holds Qf, then Kf, V and S, which wait in registers (36 KB: the
// registers set the blocks per CU).  The carried read is summed apart from the
// chunk's own and added once: one 128-term chain of fp32 sums is 1.4 x less exact
// (relative error of y against float64 3.9e-7, apart 2.6e-7).  215 us for 550 MB and
// 15 GFLOP issued (202 us with three MFMAs per product and __expf).
constexpr int OUT_THREADS = 256, OUT_ROWS = CH * 64 / OUT_THREADS;
constexpr size_t OUT_SMEM = TILE * sizeof(float2) + (4 + 1) * CH * sizeof(float);

template <int DT>
__global__ void __launch_bounds__(OUT_THREADS, 2) pc_output_kernel(qpam_pc_args a, int n) {
    extern __shared__ __align__(16) float2 smem[];
    float2 *sX = smem;
    float *sTot = reinterpret_cast<float *>(sX + TILE), *sLast = sTot + 4 * CH;
    if (Pos<OUT_ROWS>::past(a, n)) return;
    const Pos<OUT_ROWS> p(a, n);
    const int w = p.grp, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4, t = 16 * w + l16;
    const bool active = 16 * w < p.valid;
    Four q[DT];  // this lane's query row
    float2 xv[OUT_ROWS];
    {
        float2 xq[OUT_ROWS], xk[OUT_ROWS];
        float gam[OUT_ROWS], cs[OUT_ROWS];
        load_gamma<OUT_ROWS>(gam, p, a);
        load_rows<OUT_ROWS>(xq, p, a.q, p.at(a.q_sb, a.q_sh, a.q_st), a.q_st, a.dtype);
        load_rows<OUT_ROWS>(xk, p, a.k, p.at(a.k_sb, a.k_sh, a.k_st), a.k_st, a.dtype);
        load_rows<OUT_ROWS>(xv, p, a.v, p.at(a.v_sb, a.v_sh, a.v_st), a.v_st, a.v_dtype);
        prefix<OUT_ROWS>(p, gam, a.g_dtype, cs, sTot, sLast);
#pragma unroll
        for (int r = 0; r < OUT_ROWS; ++r)
            sX[p.row(r) * CP + p.j] = keep(p.ok(r), widen(xq[r], a.dtype), expf(fmaxf(cs[r], CUM_FLOOR)) * a.q_scale);
        // a wave stages exactly the rows it reads: its own LDS order before and after the reads,
        // and the block's barrier once K has taken the tile
        static_assert(OUT_ROWS == 16, "a wave's staged rows are its query tile");
        wave_lds_order();
#pragma unroll
        for (int k = 0; k < DT; ++k) q[k] = row4(sX, t, 16 * k + 4 * g);
        wave_lds_order();
#pragma unroll
        for (int r = 0; r < OUT_ROWS; ++r)
            sX[p.row(r) * CP + p.j] = keep(p.ok(r), widen(xk[r], a.dtype), expf(-fmaxf(cs[r], CUM_FLOOR)));
    }
    __syncthreads();

    floatx4 pr[4], pi[4];  // P[t][s], s = 16 st + 4 g + r
    if (active) {
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            if (st > w) continue;
            Plain x;  // sum_j conj(K[s][j]) Q[t][j]
            pz(x);
#pragma unroll
            for (int k = 0; k < DT; ++k) {
                const Four kk = row4(sX, 16 * st + l16, 16 * k + 4 * g);
#pragma unroll
                for (int r = 0; r < 4; ++r) pstep_ca(x, kk.re[r], kk.im[r], q[k].re[r], q[k].im[r]);
            }
            pr[st] = x.re;
            pi[st] = x.im;
            if (st == w) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (4 * g + r > l16) pr[st][r] = pi[st][r] = 0.f;
            }
        }
    }
    // the entering state waits in registers while V takes K's tile (lane = column)
    float2 xs[OUT_ROWS];
    const bool carry = p.t0 > 0;
    if (carry) load_state<OUT_ROWS>(xs, p, a.x + p.cc * a.d * a.d * 2, a.d);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < OUT_ROWS; ++r) sX[p.row(r) * CP + p.j] = keep(p.ok(r), widen(xv[r], a.v_dtype));
    __syncthreads();

    Plain y[DT];
#pragma unroll
    for (int it = 0; it < DT; ++it) pz(y[it]);
    if (active) {
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            if (st > w) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int it = 0; it < DT; ++it) {
                    const float2 v = sX[(16 * st + 4 * g + r) * CP + 16 * it + l16];
                    pstep(y[it], pr[st][r], pi[st][r], v.x, v.y);
                }
        }
    }
    floatx4 yr[DT], yi[DT];
#pragma unroll
    for (int it = 0; it < DT; ++it) yr[it] = y[it].re, yi[it] = y[it].im;
    if (carry) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < OUT_ROWS; ++r) sX[p.row(r) * CP + p.j] = keep(p.jv && p.row(r) < a.d, xs[r]);
        __syncthreads();
        if (active) {
#pragma unroll
            for (int it = 0; it < DT; ++it) pz(y[it]);
#pragma unroll
            for (int k = 0; k < DT; ++k)
#pragma unroll
                for (int it = 0; it < DT; ++it) {
                    const Four s = row4(sX, 16 * it + l16, 16 * k + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) pstep(y[it], q[k].re[r], q[k].im[r], s.re[r], s.im[r]);
                }
#pragma unroll
            for (int it = 0; it < DT; ++it) yr[it] += y[it].re, yi[it] += y[it].im;
        }
    }
    if (!active) return;
    const int64_t yo = ((int64_t)(p.b * a.H + p.h) * a.T + p.t0) * a.d * 2;
#pragma unroll
    for (int it = 0; it < DT; ++it) {
        const floatx4 re = yr[it], im = yi[it];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int tr = 16 * w + 4 * g + r, i = 16 * it + l16;
            if (tr < p.valid && i < a.d) st_c(a.y, yo, 2u * ((unsigned)tr * (unsigned)a.d + i), make_float2(re[r], im[r]), a.dtype);
        }
    }
}

// -------------------------------------------------------------- pc_grad --
// dq, dk, dv and dgamma of one chunk: a block of 8 waves with Qf, Kf, V and dY in
// LDS (148 KB, one block per CU).  Waves 0-3 take query tile w, waves 4-7 key tile
// w; a SIMD holds one of each, so its causal work does not depend on w:
//   query: dP = tril(dY V^H), dQ = dP Kf + dY conj(S), and of key tile w
//          dK2 = V conj(G),
//   key:   P, dP, dV = P^H dY + W G^T, dK1 = dP^H Qf,
// with S the entering state and G the gradient of the state after the chunk, which
// wait in registers and take V's and dY's tiles after the score products, W then Kf's.
// The four results replace the tiles, and each lane finishes its own channel and
// steps as the fold's backward: dq = dQ e^{L} q_scale, dk = dK1 e^{-L} + dK2 e^{L_last - L},
//   dL_t = Re(conj(Qf) dQ) - Re(conj(Kf) dK1) - Re(conj(W) dK2),
//   dL_last += sum_t Re(conj(W) dK2) + E sum_i Re(conj(S) G),
// masked where the prefix sat below -30, summed from the chunk's end and divided
// by gamma where gamma >= 1e-6.  All sums run in a fixed order; those of dL, whose
// terms cancel, in 64 bits (dgamma's distance from float64 0.96, in fp32 1.02 of that
// with three-MFMA products; the step's time is the same).  647 us for 1.0 GB
// and 40 GFLOP issued (604 us with three MFMAs per product, G scaled by E and Kf in W's place).
constexpr int GR_THREADS = 512, GR_ROWS = CH * 64 / GR_THREADS, GR_GROUPS = GR_THREADS / 64;
constexpr size_t GR_SMEM = 4 * TILE * sizeof(float2) + (5 * GR_GROUPS + 1) * CH * sizeof(float);

template <int DT>
__global__ void __launch_bounds__(GR_THREADS, 2) pc_grad_kernel(qpam_pc_args a, int n) {
    extern __shared__ __align__(16) float2 smem[];
    float2 *sQ = smem, *sK = sQ + TILE, *sV = sK + TILE, *sY = sV + TILE;
    float *sTot = reinterpret_cast<float *>(sY + TILE), *sLast = sTot + GR_GROUPS * CH;
    double *sW = reinterpret_cast<double *>(sLast + CH), *sD = sW + GR_GROUPS * CH;
    if (Pos<GR_ROWS>::past(a, n)) return;
    const Pos<GR_ROWS> p(a, n);
    const int64_t so = (int64_t)a.T * a.d * 2;
    float cs[GR_ROWS], Llast;
    {
        float gam[GR_ROWS];
        float2 xq[GR_ROWS], xk[GR_ROWS], xv[GR_ROWS], xy[GR_ROWS];
        load_gamma<GR_ROWS>(gam, p, a);
        load_rows<GR_ROWS>(xq, p, a.q, p.at(a.q_sb, a.q_sh, a.q_st), a.q_st, a.dtype);
        load_rows<GR_ROWS>(xk, p, a.k, p.at(a.k_sb, a.k_sh, a.k_st), a.k_st, a.dtype);
        load_rows<GR_ROWS>(xv, p, a.v, p.at(a.v_sb, a.v_sh, a.v_st), a.v_st, a.v_dtype);
        load_rows<GR_ROWS>(xy, p, a.dy, p.at(a.H * so, so, 2 * a.d), 2 * a.d, a.dtype);
        Llast = prefix<GR_ROWS>(p, gam, a.g_dtype, cs, sTot, sLast);
#pragma unroll
        for (int r = 0; r < GR_ROWS; ++r) {
            const float L = fmaxf(cs[r], CUM_FLOOR), al = expf(L) * a.q_scale, be = expf(-L);
            const int o = p.row(r) * CP + p.j;
            sQ[o] = keep(p.ok(r), widen(xq[r], a.dtype), al);
            sK[o] = keep(p.ok(r), widen(xk[r], a.dtype), be);
            sV[o] = keep(p.ok(r), widen(xv[r], a.v_dtype));
            sY[o] = keep(p.ok(r), widen(xy[r], a.dtype));
        }
    }
    __syncthreads();
    // S and G of the lane's column and rows, in flight behind the score products
    float2 xs[GR_ROWS], xg[GR_ROWS];
    load_state<GR_ROWS>(xs, p, a.s_in + p.cc * a.d * a.d * 2, a.d);
    load_state<GR_ROWS>(xg, p, a.x + p.cc * a.d * a.d * 2, a.d);
    const int w = p.grp & 3, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4, own = 16 * w + l16;
    const bool qside = p.grp < 4, active = 16 * w < p.valid;
    const int last = (p.valid - 1) >> 4;  // last row tile with steps
    Four own_a[DT], own_v[DT];  // query: the dY and V rows of step `own`; key (own_a): its rows of K and V, then of W
    floatx4 vr[DT], vi[DT];  // key: dV; query (later): dK2
    Plain acc[DT];           // the chunk's own dQ (query) or dK1 (key)
#pragma unroll
    for (int k = 0; k < DT; ++k) pz(acc[k]), vr[k] = vi[k] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (active) {
        if (qside) {
#pragma unroll
            for (int k = 0; k < DT; ++k) own_a[k] = row4(sY, own, 16 * k + 4 * g);
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                if (st > w) continue;
                Plain x;  // dP[t][s], lane t = own, s = 16 st + 4 g + r
                pz(x);
#pragma unroll
                for (int k = 0; k < DT; ++k) {
                    const Four v = row4(sV, 16 * st + l16, 16 * k + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) pstep_ca(x, v.re[r], v.im[r], own_a[k].re[r], own_a[k].im[r]);
                }
                floatx4 re = x.re, im = x.im;
                if (st == w) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (4 * g + r > l16) re[r] = im[r] = 0.f;
                }
#pragma unroll
                for (int r = 0; r < 4; ++r)  // dQ^T[j][t] += K[s][j] dP[t][s]
#pragma unroll
                    for (int jt = 0; jt < DT; ++jt) {
                        const float2 k = sK[(16 * st + 4 * g + r) * CP + 16 * jt + l16];
                        pstep(acc[jt], k.x, k.y, re[r], im[r]);
                    }
            }
#pragma unroll
            for (int k = 0; k < DT; ++k) own_v[k] = row4(sV, own, 16 * k + 4 * g);
        } else {
            // X[t][s] = A[t] . conj(B[s]) for t >= s (t = 16 tt + 4 g + r, lane s = own), then
            // acc^T[i][s] += C[t][i] conj(X[t][s])
            const auto side = [&](const float2 *A, const float2 *B, const float2 *C) {
#pragma unroll
                for (int k = 0; k < DT; ++k) own_a[k] = row4(B, own, 16 * k + 4 * g);
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) {
                    if (tt < w || tt > last) continue;
                    Plain x;
                    pz(x);
#pragma unroll
                    for (int k = 0; k < DT; ++k) {
                        const Four q = row4(A, 16 * tt + l16, 16 * k + 4 * g);
#pragma unroll
                        for (int r = 0; r < 4; ++r) pstep_cb(x, q.re[r], q.im[r], own_a[k].re[r], own_a[k].im[r]);
                    }
                    floatx4 re = x.re, im = x.im;
                    if (tt == w) {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (l16 > 4 * g + r) re[r] = im[r] = 0.f;
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int it = 0; it < DT; ++it) {
                            const float2 d = C[(16 * tt + 4 * g + r) * CP + 16 * it + l16];
                            pstep_cb(acc[it], d.x, d.y, re[r], im[r]);
                        }
                }
            };
            side(sQ, sK, sY);  // P, dV = P^H dY
#pragma unroll
            for (int k = 0; k < DT; ++k) vr[k] = acc[k].re, vi[k] = acc[k].im, pz(acc[k]);
            side(sY, sV, sQ);  // dP, dK1 = dP^H Q
        }
    }
    float2 kf[GR_ROWS];  // k of the lane's steps again (from the caches)
    load_rows<GR_ROWS>(kf, p, a.k, p.at(a.k_sb, a.k_sh, a.k_st), a.k_st, a.dtype);
    __syncthreads();
    // every tile is consumed: S, G and W take V's, dY's and K's, the chunk's own dQ and
    // dK1 then Q's and W's; the carried products are summed apart and added (as in pc_output)
    double wpart = 0.;  // sum_i Re(conj(S) G) of the lane's rows
#pragma unroll
    for (int r = 0; r < GR_ROWS; ++r) {
        const int o = p.row(r) * CP + p.j;
        const bool ok = p.jv && p.row(r) < a.d;
        xs[r] = keep(ok, xs[r]);
        xg[r] = keep(ok, xg[r]);
        wpart += xs[r].x * xg[r].x + xs[r].y * xg[r].y;
        sV[o] = xs[r];
        sY[o] = xg[r];
        sK[o] = keep(p.ok(r), widen(kf[r], a.dtype), __expf(Llast - fmaxf(cs[r], CUM_FLOOR)));
    }
    wpart *= __expf(Llast);
    if (qside) {
#pragma unroll
        for (int k = 0; k < DT; ++k) put4(sQ, own, 16 * k + 4 * g, acc[k].re, acc[k].im);
    }
    __syncthreads();
    if (!qside) {  // a lane replaces only what it has read itself
#pragma unroll
        for (int k = 0; k < DT; ++k) {
            own_a[k] = row4(sK, own, 16 * k + 4 * g);
            put4(sK, own, 16 * k + 4 * g, acc[k].re, acc[k].im);
        }
    }
#pragma unroll
    for (int k = 0; k < DT; ++k) pz(acc[k]);
    if (active) {
        if (qside) {
            // dQ^T[j][t] += conj(S[i][j]) dY[t][i], then dK2^T[j][s] = conj(G[i][j]) V[s][i]
            const auto carried = [&](const float2 *m, const Four (&own_x)[DT]) {
#pragma unroll
                for (int k = 0; k < DT; ++k)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int jt = 0; jt < DT; ++jt) {
                            const float2 e = m[(16 * k + 4 * g + r) * CP + 16 * jt + l16];
                            pstep_ca(acc[jt], e.x, e.y, own_x[k].re[r], own_x[k].im[r]);
                        }
            };
            carried(sV, own_a);
#pragma unroll
            for (int k = 0; k < DT; ++k) {
                const Four x = row4(sQ, own, 16 * k + 4 * g);
                const floatx4 xr = {x.re[0], x.re[1], x.re[2], x.re[3]}, xi = {x.im[0], x.im[1], x.im[2], x.im[3]};
                put4(sQ, own, 16 * k + 4 * g, xr + acc[k].re, xi + acc[k].im);
                pz(acc[k]);
            }
            carried(sY, own_v);
#pragma unroll
            for (int k = 0; k < DT; ++k) vr[k] = acc[k].re, vi[k] = acc[k].im;
        } else {
#pragma unroll
            for (int k = 0; k < DT; ++k)
#pragma unroll
                for (int it = 0; it < DT; ++it) {
                    const Four gg = row4(sY, 16 * it + l16, 16 * k + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r)  // dV^T[i][s] += G[i][j] W[s][j]
                        pstep(acc[it], gg.re[r], gg.im[r], own_a[k].re[r], own_a[k].im[r]);
                }
#pragma unroll
            for (int k = 0; k < DT; ++k) vr[k] += acc[k].re, vi[k] += acc[k].im;
        }
    }
    // and q and gamma
    float gam[GR_ROWS];
    float2 qf[GR_ROWS];
    load_gamma<GR_ROWS>(gam, p, a);
    load_rows<GR_ROWS>(qf, p, a.q, p.at(a.q_sb, a.q_sh, a.q_st), a.q_st, a.dtype);
    __syncthreads();
    // dK2 -> sY (query waves), dV -> sV (key waves); inactive row tiles are never read
#pragma unroll
    for (int k = 0; k < DT; ++k) put4(qside ? sY : sV, own, 16 * k + 4 * g, vr[k], vi[k]);
    __syncthreads();
    float dL[GR_ROWS];
    const int64_t oo = ((int64_t)(p.b * a.H + p.h) * a.T + p.t0) * a.d;  // contiguous gradients
#pragma unroll
    for (int r = 0; r < GR_ROWS; ++r) {
        const int o = p.row(r) * CP + p.j;
        dL[r] = 0.f;
        if (!p.ok(r)) continue;
        const float2 dq = sQ[o], dk1 = sK[o], dk2 = sY[o], dv = sV[o];
        const float2 xq = widen(qf[r], a.dtype), xk = widen(kf[r], a.dtype);
        const float L = fmaxf(cs[r], CUM_FLOOR), al = expf(L) * a.q_scale, be = expf(-L), ta = __expf(Llast - L);
        const float wdk = ta * (xk.x * dk2.x + xk.y * dk2.y);
        dL[r] = al * (xq.x * dq.x + xq.y * dq.y) - be * (xk.x * dk1.x + xk.y * dk1.y) - wdk;
        wpart += wdk;
        const int64_t e = 2 * (oo + p.row(r) * a.d);
        st_c(a.dq, e, 2u * p.j, make_float2(dq.x * al, dq.y * al), a.dtype);
        st_c(a.dk, e, 2u * p.j, make_float2(dk1.x * be + dk2.x * ta, dk1.y * be + dk2.y * ta), a.dtype);
        st_c(a.dv, e, 2u * p.j, dv, a.v_dtype);
    }
    sW[p.grp * CH + p.j] = wpart;
    __syncthreads();
    double dlast = 0.;
    for (int q = 0; q < GR_GROUPS; ++q) dlast += sW[q * CH + p.j];
    double run = 0., suf[GR_ROWS];
#pragma unroll
    for (int r = GR_ROWS - 1; r >= 0; --r) {
        const double d = dL[r] + (p.row(r) == p.valid - 1 ? dlast : 0.);
        run += (p.ok(r) && cs[r] >= CUM_FLOOR) ? d : 0.;
        suf[r] = run;
    }
    sD[p.grp * CH + p.j] = run;
    __syncthreads();
    double later = 0.;
    for (int q = GR_GROUPS - 1; q > p.grp; --q) later += sD[q * CH + p.j];
#pragma unroll
    for (int r = 0; r < GR_ROWS; ++r) {
        if (!p.ok(r)) continue;
        const float gv = widen(gam[r], a.g_dtype), v = gv >= GAMMA_FLOOR ? (float)(suf[r] + later) / gv : 0.f;
        const int64_t e = oo + p.row(r) * a.d;
        if (a.g_dtype == QPAM_BF16) (static_cast<unsigned short *>(a.dgamma) + e)[(unsigned)p.j] = (unsigned short)pack_bf16x2(v, v);
        else (static_cast<float *>(a.dgamma) + e)[(unsigned)p.j] = v;
    }
}

// complex elements are read and written whole: 8-byte (fp32) or 4-byte (bf16) accesses
bool whole(const void *p, int dt) { return (uintptr_t)p % (dt == QPAM_BF16 ? 4 : 8) == 0; }

int validate(const qpam_pc_args *a, const char *who) {
    QPAM_REQUIRE(a != nullptr, "%s: null args", who);
    QPAM_REQUIRE(a->B > 0 && a->H > 0 && a->T > 0, "%s: B, H, T must be positive", who);
    QPAM_REQUIRE(a->d >= 1 && a->d <= 64, "%s: head_dim must be in 1..64", who);
    QPAM_REQUIRE(a->chunk >= 1 && a->chunk <= CH, "%s: chunk must be in 1..%d", who, CH);
    for (int dt : {a->dtype, a->v_dtype, a->g_dtype})
        QPAM_REQUIRE(dt == QPAM_F32 || dt == QPAM_BF16, "%s: dtypes must be QPAM_F32 or QPAM_BF16", who);
    QPAM_REQUIRE(a->q && a->k && a->v && a->gamma && a->x && a->atot, "%s: q, k, v, gamma, x and atot are required", who);
    QPAM_REQUIRE(a->B * a->H < (1ll << 31) && a->T < (1ll << 31) &&
                     a->B * a->H * ((a->T + a->chunk - 1) / a->chunk) < (1ll << 31),
                 "%s: grid too large", who);
    const auto pairs = [](const void *p, int dt, int64_t s0, int64_t s1, int64_t s2) {
        return ((s0 | s1 | s2) & 1) == 0 && whole(p, dt);
    };
    QPAM_REQUIRE(pairs(a->q, a->dtype, a->q_sb, a->q_sh, a->q_st) && pairs(a->k, a->dtype, a->k_sb, a->k_sh, a->k_st) &&
                     pairs(a->v, a->v_dtype, a->v_sb, a->v_sh, a->v_st) && whole(a->x, QPAM_F32),
                 "%s: complex elements of q, k, v and x must be aligned", who);
    return QPAM_OK;
}

template <typename K>
int launch(K kernel, size_t smem, int threads, const qpam_pc_args &a, int n, hipStream_t s, const char *what) {
    QPAM_CHECK_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    const int64_t items = a.B * a.H * n;
    const dim3 grid((unsigned)(items < GRID_X ? items : GRID_X), (unsigned)((items + GRID_X - 1) / GRID_X));
    hipLaunchKernelGGL(kernel, grid, dim3(threads), smem, s, a, n);
    return launch_status(what);
}

int scan(const qpam_pc_args &a, int n, const float *init, float *fin, int reverse, void *stream) {
    qpam_pc_scan_args s{};
    s.N = a.B * a.H;
    s.n = n;
    s.d = a.d;
    s.x = a.x;  // in place: a lane reads two chunks ahead of its own writes
    s.out = a.x;
    s.a = a.atot;
    s.init = init;
    s.fin = fin;
    s.reverse = reverse;
    return qpam_pc_scan(&s, stream);
}

}  // namespace
}  // namespace qpam

using namespace qpam;

extern "C" int qpam_pc_fwd(const qpam_pc_args *a, void *stream) {
    int st = validate(a, "qpam_pc_fwd");
    if (st) return st;
    QPAM_REQUIRE(a->y && a->s_fin, "qpam_pc_fwd: y and s_fin are required");
    QPAM_REQUIRE(whole(a->y, a->dtype) && whole(a->s_fin, QPAM_F32),
                 "qpam_pc_fwd: complex elements of y and s_fin must be aligned");
    const int n = (int)((a->T + a->chunk - 1) / a->chunk);
    hipStream_t s = (hipStream_t)stream;
    st = a->d > 32 ? launch(pc_state_kernel<4, false>, ST_SMEM, ST_THREADS, *a, n, s, "pc_state_kernel")
                   : launch(pc_state_kernel<2, false>, ST_SMEM, ST_THREADS, *a, n, s, "pc_state_kernel");
    if (st) return st;
    st = scan(*a, n, nullptr, a->s_fin, 0, stream);
    if (st) return st;
    return a->d > 32 ? launch(pc_output_kernel<4>, OUT_SMEM, OUT_THREADS, *a, n, s, "pc_output_kernel")
                     : launch(pc_output_kernel<2>, OUT_SMEM, OUT_THREADS, *a, n, s, "pc_output_kernel");
}

extern "C" int qpam_pc_bwd(const qpam_pc_args *a, void *stream) {
    int st = validate(a, "qpam_pc_bwd");
    if (st) return st;
    QPAM_REQUIRE(a->s_in && a->dy && a->dq && a->dk && a->dv && a->dgamma,
                 "qpam_pc_bwd: s_in, dy, dq, dk, dv and dgamma are required");
    QPAM_REQUIRE(whole(a->s_in, QPAM_F32) && whole(a->dy, a->dtype) && whole(a->dfin, QPAM_F32) && whole(a->dq, a->dtype) &&
                     whole(a->dk, a->dtype) && whole(a->dv, a->v_dtype),
                 "qpam_pc_bwd: complex elements of s_in, dy, dfin, dq, dk and dv must be aligned");
    const int n = (int)((a->T + a->chunk - 1) / a->chunk);
    hipStream_t s = (hipStream_t)stream;
    st = a->d > 32 ? launch(pc_state_kernel<4, true>, ST_SMEM, ST_THREADS, *a, n, s, "pc_state_kernel")
                   : launch(pc_state_kernel<2, true>, ST_SMEM, ST_THREADS, *a, n, s, "pc_state_kernel");
    if (st) return st;
    st = scan(*a, n, a->dfin, nullptr, 1, stream);
    if (st) return st;
    return a->d > 32 ? launch(pc_grad_kernel<4>, GR_SMEM, GR_THREADS, *a, n, s, "pc_grad_kernel")
                     : launch(pc_grad_kernel<2>, GR_SMEM, GR_THREADS, *a, n, s, "pc_grad_kernel");
}
