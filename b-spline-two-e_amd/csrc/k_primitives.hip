// k_primitives.hip -- per-interval primitives of the R^k build.
//
// B-spline values: the k splines that are non-zero on interval v are
// evaluated together at a point by the Cox-de Boor triangle (de Boor,
// A Practical Guide to Splines, BSPLVB), from the same differences
// d_p(j) = t(i+j) - x and d_m(j) = x - t(i+1-j), i = k-1+iv, that BVALUE_D
// forms (bspline_tools.f90:205-211); its per-spline recurrence (:213-220)
// gives the same values to rounding.
//
// kp_windows  (one workgroup per two columns c and chunk of multipoles): spline
//   values at the k_GL outer GL points of the columns' intervals, the local
//   pair moments there
//     P^k[v;a,c] = h_v sum_q w_q B_a B_c r_q^k,
//     Q^k[v;a,c] = h_v sum_q w_q B_a B_c / r_q^(k+1)         (mat_els.f90:413-428)
//   and, per banded pair p = (a, c), (c, a) and multipole k, the window moments
//   Pw/Qw[p][j][k] (j-th interval of p's support window), their prefix (P) and
//   suffix (Q) sums and totals.
// kp_inner  (one workgroup per interval and chunk of kc multipoles): spline
//   values at the k_GL^2 inner points of the triangle rule and the diagonal
//   cells of mat_els.f90:460-483 as the contraction over the outer points
//     D[v][uo][ui][k] = h_v sum_q (w_q B_a B_c)(r_q) * J'[k][q][ui],
//     J'[k][q][u]     = s_q / r_q^(k+1) * sum_p w_p rho_qp^k B_b B_d(rho_qp),
//   with s_q = (r_q - bp_v)/2 and rho_qp = s_q x_p + (r_q + bp_v)/2, on the
//   FP64 matrix cores, a few multipoles at a time staged in LDS.
// kw_pair_windows: the same window tables gathered from the local moments
//   Pl/Ql[v][u][k] of the U = k(k+1)/2 unordered local spline pairs u (what the
//   mixed-precision moments write).
#include <algorithm>

#include "bs2e_internal.h"
#include "bspline_device.h"

namespace bs2e {

constexpr int kPThreads = 256;
constexpr int kFewCells = 384;   // diagonal-cell workgroups

static inline unsigned blocks_for(int64_t n, int threads) { return (unsigned)((n + threads - 1) / threads); }

hipError_t allow_lds(const void* fn, size_t bytes)
{
    if (bytes <= 64 * 1024) return hipSuccess;
    return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// Which bases are accepted and which multipole chunks a caller can pin, as
// earlier layouts of the diagonal cells in LDS allowed: tables of every multipole
// of a chunk, at most 16 of them up to order 9 and 16 GL points, 4 elsewhere.
// The kernels' own tables (diag_lds_bytes, window_lds_bytes of window_shape) fit
// for every order, GL order and multipole count that this lets through; it stays
// as the line because callers meet it as a refusal.
size_t inner_lds_bytes(int64_t ks, int64_t kgl, int64_t kc)
{
    const int64_t U = ks * (ks + 1) / 2;
    if (ks <= 9 && kgl <= 16)
        return sizeof(double) * (size_t)(kgl * ks + kgl * kgl * ks + kgl + kgl * U + 2 * kgl * kgl + kc * kgl * U);
    return sizeof(double) *
           (size_t)(kgl * ks + kgl * kgl * ks + kgl + kgl * kgl + kgl * U + kc * kgl * kgl + kc * kgl * U);
}

int inner_kc(int64_t ks, int64_t kgl, int64_t K)
{
    if (ks <= 9 && kgl <= 16) {
        for (int64_t kc = std::min<int64_t>(K, 16); kc >= 1; --kc)
            if (inner_lds_bytes(ks, kgl, kc) <= kLdsPerWorkgroup) return (int)kc;
        return 0;
    }
    for (int kc : {4, 2, 1})
        if (kc <= K && inner_lds_bytes(ks, kgl, kc) <= kLdsPerWorkgroup) return kc;
    return inner_lds_bytes(ks, kgl, 1) <= kLdsPerWorkgroup ? 1 : 0;
}

// LDS of a diagonal-cell workgroup that holds the inner moments of KC
// multipoles at a time: the splines at the outer and inner points, the outer
// pair products (over the GL points padded to a multiple of four) and inner
// moments, and X and its ratio at the inner points.  All that inner_kc accepts
// fits with KC = 1.
static size_t diag_lds_bytes(int64_t ks, int64_t kgl, int64_t KC)
{
    const int64_t U = ks * (ks + 1) / 2, QP = (kgl + 3) / 4 * 4;
    return sizeof(double) * (size_t)(kgl * (1 + kgl) * ks + 2 * kgl * kgl + (KC * kgl + QP) * U);
}

// Columns and multipoles of one window workgroup.
struct WindowShape {
    int cols, kc, kchunks, n_wg;
};

// What the window workgroups read and write; pairs, Pl and Ql for the gather
// from local moments, c_first for the moments taken here.
struct WindowArgs {
    WindowShape ws;
    int n_b, n_iv, n_pairs;
    const int32_t* c_first;
    const PairInfo* pairs;
    const double *Pl, *Ql;
    double *Pw, *Qw, *PP, *QS, *Ptot, *Qtot;
};

static size_t window_lds_bytes(int64_t ks, int64_t kgl, int64_t cols, int64_t kc)
{
    const int64_t npt = (ks + cols - 1) * kgl;
    return sizeof(double) * (size_t)(npt * (ks + 1 + 2 * kc) + cols * ks * (ks + 1) * kc);
}

// The window moments of the pairs (a, c) of `cols` columns c and kc multipoles,
// and their sums.  Moments and window sums in one pass: the local moments of an
// interval in a launch of their own and a gather of the windows after it took a
// launch more, which a small build waits for (order 8, 46 splines, 5 multipoles,
// whole build 23.5 us, now 19.6; 65 splines 24.9, now 21.1); a column evaluates
// the splines of its k intervals again for that.  The local pair (ta, tc), ta <= tc, of interval c + 1 - tc is
// the pair (c - tc + ta, c) there, so a column takes every local pair once; the
// pair (c, a) has the same numbers.
template <int KS, int T>
__device__ __forceinline__ void window_columns(int wg, const WindowArgs& A, int K, int kgl,
                                               const double* __restrict__ t, const double* __restrict__ bp,
                                               const double* __restrict__ x, const double* __restrict__ w, double* lds)
{
    const WindowShape ws = A.ws;
    const int n_b = A.n_b, n_iv = A.n_iv;
    const int32_t* __restrict__ c_first = A.c_first;
    double *__restrict__ Pw = A.Pw, *__restrict__ Qw = A.Qw, *__restrict__ PP = A.PP, *__restrict__ QS = A.QS;
    double *__restrict__ Ptot = A.Ptot, *__restrict__ Qtot = A.Qtot;
    constexpr int U = KS * (KS + 1) / 2;
    const int blk = wg / ws.kchunks, k0 = (wg - blk * ws.kchunks) * ws.kc;
    const int nk = min(ws.kc, K - k0);
    const int c0 = blk * ws.cols + 1, nc = min(ws.cols, n_b + 1 - c0);
    const int iv0 = max(1, c0 + 2 - KS), npt = (min(n_iv, c0 + nc) + 1 - iv0) * kgl;
    double* sB = lds;                        // [npt][KS]
    double* sR = sB + npt * KS;              // [npt]
    double* sPow = sR + npt;                 // [npt][nk]  r^k
    double* sInv = sPow + npt * nk;          // [npt][nk]  1 / r^(k+1)
    double* sP = sInv + npt * nk;            // [nc][U][nk]
    double* sQ = sP + nc * U * nk;           // [nc][U][nk]
    const int tid = threadIdx.x;
    for (int e = tid; e < npt; e += T) {
        const int iv = iv0 + e / kgl, q = e - (iv - iv0) * kgl;
        const double lim1 = bp[iv - 1], lim2 = bp[iv];
        const double r = gl_point(0.5 * (lim2 - lim1), 0.5 * (lim2 + lim1), x[q]);
        sR[e] = r;
        splines_at<KS>(t, KS - 1 + iv, r, sB + e * KS, 1);
    }
    __syncthreads();
    for (int e = tid; e < npt * nk; e += T) {
        const int i = e / nk, k = k0 + e - i * nk;
        const double r = sR[i];
        sPow[e] = ipow_d(r, k);
        sInv[e] = 1.0 / ipow_d(r, k + 1);
    }
    __syncthreads();
    for (int e = tid; e < nc * U * nk; e += T) {
        const int cu = e / nk, kk = e - cu * nk, c = c0 + cu / U, u = cu - (c - c0) * U;
        int ta, tc;
        local_pair(u, KS, ta, tc);
        const int iv = c + 1 - tc;
        if (iv < 1 || iv > n_iv) continue;
        const int i0 = (iv - iv0) * kgl;
        double accp = 0.0, accq = 0.0;
        for (int q = 0; q < kgl; ++q) {
            const double* b = sB + (i0 + q) * KS;
            const double bb = w[q] * b[ta] * b[tc];
            accp = accp + bb * sPow[(i0 + q) * nk + kk];
            accq = accq + bb * sInv[(i0 + q) * nk + kk];
        }
        const double h = 0.5 * (bp[iv] - bp[iv - 1]);
        sP[e] = h * accp;
        sQ[e] = h * accq;
    }
    __syncthreads();
    for (int e = tid; e < 2 * nc * KS * nk; e += T) {
        int r = e / nk;
        const int kk = e - r * nk, i = r % KS;      // a = c - i
        r /= KS;
        const int c = c0 + (r >> 1), a = c - i;
        const bool mirror = r & 1;
        if (a < 1 || (mirror && i == 0)) continue;
        const int row = mirror ? c : a, col = mirror ? a : c;
        const size_t pair = (size_t)(c_first[col] + row - max(1, col + 1 - KS));
        const int v0 = max(1, c + 2 - KS), m = min(n_iv, a + 1) + 1 - v0;
        const size_t base = pair * KS * K + k0 + kk;
        const int uc = (c - c0) * U;
        double pw[KS], qw[KS];
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            pw[j] = 0.0;
            qw[j] = 0.0;
            if (j < m) {
                const int tc = c + 1 - v0 - j, u = uc + sym_local(tc - i, tc, KS);
                pw[j] = sP[u * nk + kk];
                qw[j] = sQ[u * nk + kk];
            }
        }
        double run = 0.0;
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            run += pw[j];
            Pw[base + (size_t)j * K] = pw[j];
            Qw[base + (size_t)j * K] = qw[j];
            PP[base + (size_t)j * K] = (j < m) ? run : 0.0;
        }
        Ptot[pair * K + k0 + kk] = run;
        run = 0.0;
#pragma unroll
        for (int j = KS - 1; j >= 0; --j) {
            run += qw[j];
            QS[base + (size_t)j * K] = (j < m) ? run : 0.0;
        }
        Qtot[pair * K + k0 + kk] = run;
    }
}

// The same from local moments that an earlier launch wrote, one thread per
// pair and multipole.
template <int KSMAX>
__device__ __forceinline__ void window_gather(int64_t gid, const WindowArgs& A, int K, int ks)
{
    if (gid >= (int64_t)A.n_pairs * K) return;
    const int U = ks * (ks + 1) / 2;
    const int p = (int)(gid / K), k = (int)(gid - (int64_t)p * K);
    const PairInfo pi = A.pairs[p];
    const double *__restrict__ Pl = A.Pl, *__restrict__ Ql = A.Ql;
    double *__restrict__ Pw = A.Pw, *__restrict__ Qw = A.Qw, *__restrict__ PP = A.PP, *__restrict__ QS = A.QS;
    double pw[KSMAX], qw[KSMAX];
#pragma unroll
    for (int j = 0; j < KSMAX; ++j) {
        pw[j] = 0.0;
        qw[j] = 0.0;
        if (j < pi.m) {
            const int v = pi.v0 - 1 + j;                         // 0-based interval
            const int u = sym_local(pi.a - v, pi.c - v, ks);     // local splines s - iv
            pw[j] = Pl[((size_t)v * U + u) * K + k];
            qw[j] = Ql[((size_t)v * U + u) * K + k];
        }
    }
    const size_t base = (size_t)p * ks * K + k;
    double run = 0.0;
#pragma unroll
    for (int j = 0; j < KSMAX; ++j) {
        if (j < ks) {
            run += pw[j];
            Pw[base + (size_t)j * K] = pw[j];
            Qw[base + (size_t)j * K] = qw[j];
            PP[base + (size_t)j * K] = (j < pi.m) ? run : 0.0;
        }
    }
    A.Ptot[(size_t)p * K + k] = run;
    run = 0.0;
#pragma unroll
    for (int j = KSMAX - 1; j >= 0; --j) {
        if (j < ks) {
            run += qw[j];
            QS[base + (size_t)j * K] = (j < pi.m) ? run : 0.0;
        }
    }
    A.Qtot[(size_t)p * K + k] = run;
}

template <int KS>
__global__ __launch_bounds__(kPThreads) void kp_windows(WindowArgs A, int K, int kgl, const double* __restrict__ t,
                                                        const double* __restrict__ bp, const double* __restrict__ x,
                                                        const double* __restrict__ w)
{
    extern __shared__ double lds[];
    window_columns<KS, kPThreads>((int)xcd_block(blockIdx.x, A.ws.n_wg), A, K, kgl, t, bp, x, w, lds);
}

template <int KSMAX>
__global__ __launch_bounds__(kPThreads) void kw_pair_windows(WindowArgs A, int K, int ks)
{
    window_gather<KSMAX>((int64_t)blockIdx.x * kPThreads + threadIdx.x, A, K, ks);
}

// The diagonal cells.  SYM: write Dsym[v][u1][u2][k] = D[v][u1][u2][k] +
// D[v][u2][u1][k] (what the tensor consumes) for u1 <= u2 only, the symmetric
// matrix's upper triangle, instead of D (what the sparse_6d container holds).
// Per workgroup: interval v and multipoles k0 .. k0+nk-1 (the chunks of one
// interval sit on one XCD, so the K-contiguous records of D are completed in
// one L2).
//   stage 1: splines at the outer and inner points; X_k0[q][p] =
//            s_q w_p rho^k0 / r_q^(k0+1) (from X_0 by k0 multiplications with
//            the ratio rho / r_q, so that every chunking gives the same bits);
//   stage 2: WB[q][u] = w_q B_a B_c (r_q);
// then for KC multipoles at a time
//   stage 3: J'[kk][q][u] = sum_p X_k[q][p] B_b B_d (rho_qp), the powers by
//            repeated multiplication with the ratio;
//   stage 4: per 16 x 16 tile of (uo, ui) and two multipoles, on
//            v_mfma_f64_16x16x4: D = WB^T J' (SYM: Dsym = WB^T J' + J'^T WB,
//            the two products in separate accumulators, upper-triangle tiles
//            and elements only), zero-padded to a multiple of four GL points.
// The FP64 matrix cores run at the vector rate; they are used because a tile
// reads its operands from LDS 16 times less often.  Bound by latency: the
// stages are short and wait for one another, so what counts is the number of
// workgroups a CU holds (KC as small as keeps the two multipoles of a tile
// busy: the inner moments of all multipoles at once took 104 KB of LDS at
// order 9, one workgroup per CU) and a loop body that stays in the instruction
// cache.
// WITH: the workgroups past the n_cells of the cells take the window moments,
// or gather them.
enum class With { kNothing, kMoments, kGather };

template <int KS, bool SYM, int KC, int T, With WITH>
__global__ __launch_bounds__(T) void kp_inner(int K, int kgl, int kc, int kchunks, int n_cells, WindowArgs A,
                                                      const double* __restrict__ t, const double* __restrict__ bp,
                                                      const double* __restrict__ x, const double* __restrict__ w,
                                                      double* __restrict__ D)
{
    constexpr int U = KS * (KS + 1) / 2;
    constexpr int TU = (U + 15) / 16;
    constexpr int NT = SYM ? TU * (TU + 1) / 2 : TU * TU;
    constexpr int NP = (KC + 1) / 2;         // pairs of multipoles per group
    typedef double d4_t __attribute__((ext_vector_type(4)));
    typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));
    extern __shared__ double lds[];
    if (WITH != With::kNothing && (int)blockIdx.x >= n_cells) {
        const int wg = (int)blockIdx.x - n_cells;
        if constexpr (WITH == With::kMoments) window_columns<KS, T>(wg, A, K, kgl, t, bp, x, w, lds);
        else window_gather<KS>((int64_t)wg * T + threadIdx.x, A, K, KS);
        return;
    }
    const int npt = kgl * (1 + kgl), QP = (kgl + 3) & ~3;
    double* sB = lds;                        // [kgl + kgl * kgl][KS]: outer points, then inner points
    double* sX = sB + npt * KS;              // [kgl][kgl]      X of the group's first multipole
    double* sXr = sX + kgl * kgl;            // [kgl][kgl]      rho / r_q
    double* sJ = sXr + kgl * kgl;            // [KC][kgl][U]    (read past kgl: the next rows, times a zero of sWB)
    double* sWB = sJ + KC * kgl * U;         // [QP][U]         w_q B_a B_c at r_q (zero past kgl)

    const int64_t lg = xcd_block(blockIdx.x, n_cells);
    const int v = (int)(lg / kchunks);
    const int k0 = (int)(lg - (int64_t)v * kchunks) * kc;
    const int nk = (K - k0) < kc ? (K - k0) : kc;
    const int tid = threadIdx.x;
    const double lim1 = bp[v], lim2 = bp[v + 1];
    const double h = 0.5 * (lim2 - lim1);
    const double c = 0.5 * (lim2 + lim1);
    const int i1 = KS - 1 + (v + 1);

#pragma unroll 1
    for (int e = tid; e < npt; e += T) {
        const bool inner = e >= kgl;
        const int q = inner ? e / kgl - 1 : e, pp = inner ? e - (q + 1) * kgl : 0;
        const double rq = gl_point(h, c, x[q]);
        const double rho = inner ? 0.5 * (rq - lim1) * x[pp] + 0.5 * (rq + lim1) : rq;
        splines_at<KS>(t, i1, rho, sB + e * KS, 1);
        if (inner) {
            // X_k = s_q w_p rho^k / r_q^(k+1) = X_0 (rho / r_q)^k, the same
            // multiplication sequence from k = 0 for every chunking
            const double ratio = rho / rq;
            double xk = 0.5 * (rq - lim1) * w[pp] / rq;
            for (int j = 0; j < k0; ++j) xk *= ratio;
            sX[e - kgl] = xk;
            sXr[e - kgl] = ratio;
        }
    }
    for (int e = kgl * U + tid; e < QP * U; e += T) sWB[e] = 0.0;
    __syncthreads();
#pragma unroll 1
    for (int e = tid; e < kgl * U; e += T) {
        const int q = e / U, u = e - q * U;
        int ta, tc;
        local_pair(u, KS, ta, tc);
        sWB[e] = w[q] * sB[q * KS + ta] * sB[q * KS + tc];
    }
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int li = lane & 15, lk = lane >> 4;
#pragma unroll 1
    for (int g = 0; g < nk; g += KC) {
#pragma unroll 1
        for (int e = tid; e < kgl * U; e += T) {
            const int q = e / U, u = e - q * U;
            int ta, tc;
            local_pair(u, KS, ta, tc);
            double acc[KC];
#pragma unroll
            for (int kk = 0; kk < KC; ++kk) acc[kk] = 0.0;
            const double* bq = sB + (kgl + q * kgl) * KS;
            const double* xq = sX + q * kgl;
            const double* rq = sXr + q * kgl;
#pragma unroll 2
            for (int pp = 0; pp < kgl; ++pp) {
                const double bb = bq[pp * KS + ta] * bq[pp * KS + tc];
                double xk = xq[pp];
                const double ratio = rq[pp];
#pragma unroll
                for (int kk = 0; kk < KC; ++kk) {   // (past the chunk's last multipole: not used)
                    acc[kk] += xk * bb;
                    xk *= ratio;
                }
            }
#pragma unroll
            for (int kk = 0; kk < KC; ++kk) sJ[kk * kgl * U + e] = acc[kk];
        }
        __syncthreads();
        for (int e = tid; e < kgl * kgl; e += T) {   // (read again after the next barrier)
            double xk = sX[e];
#pragma unroll
            for (int kk = 0; kk < KC; ++kk) xk *= sXr[e];
            sX[e] = xk;
        }
        const int left = nk - g;             // multipoles from this group on
#pragma unroll 1
        for (int item = wave; item < NT * NP; item += T / 64) {
            const int tile = item / NP, kk = 2 * (item - tile * NP);
            if (kk >= left) continue;
            const bool two = KC > 1 && kk + 1 < left;
            int ta, tb;
            if (SYM) {   // upper-triangle tiles, row by row
                ta = 0;
                int r = tile;
                while (r >= TU - ta) {
                    r -= TU - ta;
                    ++ta;
                }
                tb = ta + r;
            } else {
                ta = tile / TU;
                tb = tile - ta * TU;
            }
            // operand row / column of this lane (clamped: elements past U are not stored)
            const int ua = min(ta * 16 + li, U - 1), ub = min(tb * 16 + li, U - 1);
            const double* W = sWB + lk * U;
            const double* J0 = sJ + (kk * kgl + lk) * U;
            const double* J1 = KC > 1 ? J0 + kgl * U : J0;
            d4_t c0 = {0.0, 0.0, 0.0, 0.0}, c1 = c0, e0 = c0, e1 = c0;
#pragma unroll 2
            for (int q = 0; q < QP; q += 4) {
                const double a1 = W[q * U + ua], b0 = J0[q * U + ub], b1 = J1[q * U + ub];
                c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, c0, 0, 0, 0);
                if (KC > 1) c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, c1, 0, 0, 0);
                if (SYM) {
                    const double b2 = W[q * U + ub], a20 = J0[q * U + ua], a21 = J1[q * U + ua];
                    e0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a20, b2, e0, 0, 0, 0);
                    if (KC > 1) e1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a21, b2, e1, 0, 0, 0);
                }
            }
            // result row (lane >> 4) + 4 r, column lane & 15 of the tile
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int uo = ta * 16 + lk + 4 * r, ui = tb * 16 + li;
                if (uo < U && ui < U && (!SYM || uo <= ui)) {
                    double* dst = D + (((size_t)v * U + uo) * U + ui) * K + k0 + g + kk;
                    const double d0 = h * (SYM ? c0[r] + e0[r] : c0[r]), d1 = h * (SYM ? c1[r] + e1[r] : c1[r]);
                    if (two) *(d2u_t*)dst = d2u_t{d0, d1};
                    else *dst = d0;
                }
            }
        }
        __syncthreads();
    }
}

// Window prefix/suffix sums from Pw/Qw already in place (the moments were
// gathered from caller-provided containers).
__global__ __launch_bounds__(256) void kw_window_sums(int n_pairs, int K, int ks, const PairInfo* __restrict__ pairs,
                                                      const double* __restrict__ Pw, const double* __restrict__ Qw,
                                                      double* __restrict__ PP, double* __restrict__ QS,
                                                      double* __restrict__ Ptot, double* __restrict__ Qtot)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (int64_t)n_pairs * K) return;
    const int p = (int)(gid / K), k = (int)(gid - (int64_t)p * K);
    const int m = pairs[p].m;
    const size_t base = (size_t)p * ks * K + k;
    double run = 0.0;
    for (int j = 0; j < ks; ++j) {
        if (j < m) run += Pw[base + (size_t)j * K];
        PP[base + (size_t)j * K] = (j < m) ? run : 0.0;
    }
    Ptot[(size_t)p * K + k] = run;
    run = 0.0;
    for (int j = ks - 1; j >= 0; --j) {
        if (j < m) run += Qw[base + (size_t)j * K];
        QS[base + (size_t)j * K] = (j < m) ? run : 0.0;
    }
    Qtot[(size_t)p * K + k] = run;
}

// Two columns and at most four multipoles per workgroup, in equal chunks: the
// kernel is a chain of short stages (splines, powers, moments, sums), so it
// takes many small workgroups; more columns share the splines of more
// intervals, fewer give more workgroups.  Columns x multipoles, until the
// windows are done (order 9, 600 splines, 25 multipoles / order 9, 400, 17 /
// order 8, 200, 11, with the launch): 2 x 4 38 / 23 / 16 us, 1 x 4 44 / 26 / 14,
// 4 x 4 58 / 26 / 16, 8 x 4 62 / 28 / 20, 2 x 8 52 / 25 / 16, 1 x 16 48 / 37 / 15.
static WindowShape window_shape(const Plan& p)
{
    int cols = 2, kchunks = (int)((p.K + 3) / 4);
    int kc = (int)((p.K + kchunks - 1) / kchunks);
    if (window_lds_bytes(p.k_s, p.k_gl, cols, kc) > 64 * 1024) cols = 1;
    while (kc > 1 && window_lds_bytes(p.k_s, p.k_gl, cols, kc) > kLdsPerWorkgroup) --kc;
    kchunks = (int)((p.K + kc - 1) / kc);
    return {cols, kc, kchunks, (int)((p.n_b + cols - 1) / cols) * kchunks};
}

static WindowArgs window_args(const Plan& p, const DevTables& d)
{
    return {window_shape(p), (int)p.n_b, (int)p.n_iv, (int)p.n_pairs, d.c_first, d.pairs, d.Pl, d.Ql,
            d.Pw, d.Qw, d.PP, d.QS, d.Ptot, d.Qtot};
}

template <int KS>
static void launch_windows(const Plan& p, const DevTables& d, hipStream_t s)
{
    const WindowArgs A = window_args(p, d);
    const size_t lds = window_lds_bytes(KS, p.k_gl, A.ws.cols, A.ws.kc);
    if (allow_lds((const void*)kp_windows<KS>, lds) != hipSuccess) return;   // the error stays for hipGetLastError
    hipLaunchKernelGGL(kp_windows<KS>, dim3((unsigned)A.ws.n_wg), dim3(kPThreads), lds, s, A, (int)p.K, (int)p.k_gl,
                       d.t, d.bp, d.x, d.w);
}

// Multipoles that a diagonal-cell workgroup holds at a time: four; two where
// groups of four would leave CUs without a workgroup (a shorter chain: order
// 8, 41 intervals, 5 multipoles 10.1 us against 12.0), or their tables do not
// fit (then one).  Groups of eight: 0.123 ms against 0.118 at order 9, 593
// intervals, 25 multipoles; 0.088 against 0.047 at order 10, 175 intervals, 9.
static int inner_group(const Plan& p)
{
    if (p.n_iv * ((p.K + 3) / 4) > 256 && diag_lds_bytes(p.k_s, p.k_gl, 4) <= kLdsPerWorkgroup) return 4;
    return diag_lds_bytes(p.k_s, p.k_gl, 2) <= kLdsPerWorkgroup ? 2 : 1;
}

// Whole groups per workgroup, as many as leave two workgroups per CU (every
// workgroup evaluates its interval's splines): order 8, 195 intervals, 11
// multipoles in chunks of 4 18.9 us, in one chunk 23.0, of 2 25.3.
int inner_kc_used(const Plan& p)
{
    const int kmax = inner_kc(p.k_s, p.k_gl, p.K);
    if (p.inner_kc >= 1 && p.inner_kc <= kmax) return p.inner_kc;
    const int64_t KC = inner_group(p), chunks = (512 + p.n_iv - 1) / p.n_iv;
    const int64_t kc = ((p.K + chunks - 1) / chunks + KC - 1) / KC * KC;
    return (int)std::min<int64_t>(kc, std::max(kmax, 1));
}

template <int KS, bool SYM, int KC, int T, With WITH>
static void launch_inner_kc(const Plan& p, const DevTables& d, hipStream_t s)
{
    const int kc = inner_kc_used(p), kchunks = (int)((p.K + kc - 1) / kc);
    const int n_cells = (int)(p.n_iv * kchunks);
    const WindowArgs A = window_args(p, d);
    size_t lds = diag_lds_bytes(KS, p.k_gl, KC);
    unsigned n_wg = (unsigned)n_cells;
    if (WITH == With::kMoments) {
        lds = std::max(lds, window_lds_bytes(KS, p.k_gl, A.ws.cols, A.ws.kc));
        n_wg += (unsigned)A.ws.n_wg;
    }
    if (WITH == With::kGather) n_wg += blocks_for(p.n_pairs * p.K, T);
    const auto fn = kp_inner<KS, SYM, KC, T, WITH>;
    if (allow_lds((const void*)fn, lds) != hipSuccess) return;   // the error stays for hipGetLastError
    hipLaunchKernelGGL(fn, dim3(n_wg), dim3(T), lds, s, (int)p.K, (int)p.k_gl, kc, kchunks, n_cells, A, d.t,
                       d.bp, d.x, d.w, d.D);
}

template <int KS, bool SYM, int T, With WITH>
static void launch_inner_threads(const Plan& p, const DevTables& d, hipStream_t s)
{
    const int KC = inner_group(p);
    if (KC == 4) launch_inner_kc<KS, SYM, 4, T, WITH>(p, d, s);
    else if (KC == 2) launch_inner_kc<KS, SYM, 2, T, WITH>(p, d, s);
    else launch_inner_kc<KS, SYM, 1, T, WITH>(p, d, s);
}

// Small builds whose cells give a CU one workgroup or little more (kFewCells)
// take them with twice the threads: nothing else covers a stage's latency there.
// Whole builds, 512 threads against 256: order 8, 46 splines, 5 multipoles (120
// workgroups) 17.0 / 19.7 us, order 16, 73, 3 (116) 74 / 95, order 9, 82, 16 (304)
// 51.1 / 54.1, order 10, 114, 9 (321) 70-72 / 75, order 12, 85, 9 (370) 75.3 / 80.7;
// but order 8, 160, 9 (465) 82.0 / 80.6 and order 5, 189, 12 (561) 52.0 / 50.3.
// Beside the fill on a second stream they would take its wave slots: order 8, 200
// splines 183 / 151 us.
template <int KS, bool SYM, With WITH>
static void launch_inner(const Plan& p, const DevTables& d, hipStream_t s)
{
    if constexpr (WITH != With::kNothing) {
        const int64_t kc = inner_kc_used(p);
        if (p.n_iv * ((p.K + kc - 1) / kc) <= kFewCells)
            return launch_inner_threads<KS, SYM, 2 * kPThreads, WITH>(p, d, s);
    }
    launch_inner_threads<KS, SYM, kPThreads, WITH>(p, d, s);
}

template <int KS>
static void launch_inner_sym(const Plan& p, const DevTables& d, hipStream_t s)
{
    launch_inner<KS, true, With::kNothing>(p, d, s);
}

template <int KS>
static void launch_inner_plain(const Plan& p, const DevTables& d, hipStream_t s)
{
    launch_inner<KS, false, With::kNothing>(p, d, s);
}

template <int KS>
static void launch_inner_windows(const Plan& p, const DevTables& d, hipStream_t s)
{
    launch_inner<KS, true, With::kMoments>(p, d, s);
}

template <int KS>
static void launch_inner_gather(const Plan& p, const DevTables& d, hipStream_t s)
{
    launch_inner<KS, true, With::kGather>(p, d, s);
}

#define BS2E_ORDER_SWITCH(FN)                                                                                \
    switch (p.k_s) {                                                                                         \
        case 2: FN<2>(p, d, s); break;                                                                       \
        case 3: FN<3>(p, d, s); break;                                                                       \
        case 4: FN<4>(p, d, s); break;                                                                       \
        case 5: FN<5>(p, d, s); break;                                                                       \
        case 6: FN<6>(p, d, s); break;                                                                       \
        case 7: FN<7>(p, d, s); break;                                                                       \
        case 8: FN<8>(p, d, s); break;                                                                       \
        case 9: FN<9>(p, d, s); break;                                                                       \
        case 10: FN<10>(p, d, s); break;                                                                     \
        case 11: FN<11>(p, d, s); break;                                                                     \
        case 12: FN<12>(p, d, s); break;                                                                     \
        case 13: FN<13>(p, d, s); break;                                                                     \
        case 14: FN<14>(p, d, s); break;                                                                     \
        case 15: FN<15>(p, d, s); break;                                                                     \
        case 16: FN<16>(p, d, s); break;                                                                     \
        default: return hipErrorInvalidValue;                                                                \
    }

hipError_t launch_windows(const Plan& p, const DevTables& d, hipStream_t s)
{
    BS2E_ORDER_SWITCH(launch_windows)
    return hipGetLastError();
}

hipError_t launch_diag_cells(const Plan& p, const DevTables& d, hipStream_t s, bool symmetrised)
{
    if (symmetrised) {
        BS2E_ORDER_SWITCH(launch_inner_sym)
    } else {
        BS2E_ORDER_SWITCH(launch_inner_plain)
    }
    return hipGetLastError();
}

hipError_t launch_windows_and_cells(const Plan& p, const DevTables& d, bool gather, hipStream_t s)
{
    if (gather) {
        BS2E_ORDER_SWITCH(launch_inner_gather)
    } else {
        BS2E_ORDER_SWITCH(launch_inner_windows)
    }
    return hipGetLastError();
}

template <int KSMAX>
static void launch_kw(const Plan& p, const DevTables& d, hipStream_t s)
{
    hipLaunchKernelGGL(kw_pair_windows<KSMAX>, dim3(blocks_for(p.n_pairs * p.K, kPThreads)), dim3(kPThreads), 0, s,
                       window_args(p, d), (int)p.K, (int)p.k_s);
}

hipError_t launch_pair_windows(const Plan& p, const DevTables& d, hipStream_t s)
{
    if (p.k_s <= 6) launch_kw<6>(p, d, s);
    else if (p.k_s <= 8) launch_kw<8>(p, d, s);
    else if (p.k_s <= 10) launch_kw<10>(p, d, s);
    else if (p.k_s <= 12) launch_kw<12>(p, d, s);
    else launch_kw<16>(p, d, s);
    return hipGetLastError();
}

hipError_t launch_window_sums(const Plan& p, const DevTables& d, hipStream_t s)
{
    const int64_t n = p.n_pairs * p.K;
    hipLaunchKernelGGL(kw_window_sums, dim3(blocks_for(n, 256)), dim3(256), 0, s, (int)p.n_pairs, (int)p.K,
                       (int)p.k_s, d.pairs, d.Pw, d.Qw, d.PP, d.QS, d.Ptot, d.Qtot);
    return hipGetLastError();
}

}  // namespace bs2e
