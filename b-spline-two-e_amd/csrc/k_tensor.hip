// k_tensor.hip -- the banded R^k tensor (sparse_array_tools.f90:452-493).
//
// For banded pairs p = (a,c) (electron 1) and q = (b,d) (electron 2) with
// support windows W_p, W_q (intervals), the reference accumulates
//   R^k(a,b,c,d) = sum_{v<w} P^k[v;p] Q^k[w;q] + sum_{v>w} Q^k[v;p] P^k[w;q]
//                + sum_{v in W_p and W_q} ( D^k[v;p,q] + D^k[v;q,p] )
// over the nnz4^2 off-diagonal products and the nnz6 diagonal cells
// (sparse_array_tools.f90:472-488).  Because the windows are contiguous:
//   * W_p entirely left of W_q :  R = Ptot[p] * Qtot[q]            (rank one)
//   * W_p entirely right of W_q:  R = Qtot[p] * Ptot[q]            (rank one)
//   * in general                :  R = sum_{w in W_q} Qw_q(w) PP_p(w-1)
//                                     + Pw_q(w) QS_p(w+1) + sum_v Dsym[v;p,q]
// with PP_p / QS_p the prefix / suffix sums of P / Q over W_p and
// Dsym[v] = D[v] + D[v]^T the symmetrised diagonal cell.
//
// Two kernels write disjoint elements, each element exactly once:
//   * k3_far : two rows x one column chunk of rank-one products (the pairs'
//     windows do not overlap), streamed with non-temporal stores.  Bound by
//     the FP64 store of R: 8 bytes per integral.
//   * k3_near: the elements whose pairs share a support interval (a few
//     percent of each row).  R(a,b,c,d) = R(c,b,a,d) = R(a,d,c,b) = R(b,a,d,c),
//     so one workgroup per row (a,c), a <= c, evaluates its columns (b,d),
//     b <= d, that are not before the row and stores each value into all the
//     equal elements.  With W_p = [lo, hi], for column q:
//       R = Qtot_p * sum_{w in W_q, w < lo} P_q(w)
//         + Ptot_p * sum_{w in W_q, w > hi} Q_q(w)
//         + sum_{w in W_p and W_q} Q_q(w) PP_p(w-1) + P_q(w) QS_p(w+1) + Dsym[w; p, q]
//     (the general formula with PP_p = 0 left of W_p and Ptot_p right of it,
//     QS_p = Qtot_p left of W_p and 0 right of it); the first two sums are
//     q's own prefix / suffix sums.  It runs beside k3_far: on a second
//     stream, or for small tensors in one launch with it (k3_fill).
#include <algorithm>

#include "bs2e_internal.h"

namespace bs2e {

constexpr int kThreads = 256;

// Rounded-up 32-bit reciprocal of n (0 for n = 1): the upper half of its
// product with x is x / n exactly for x < 2^32 / n.
static unsigned recip32(int64_t n) { return n > 1 ? (unsigned)((((uint64_t)1 << 32) + n - 1) / n) : 0; }

// LDS of a near workgroup (row p, window length m):
//   PPx[i][k], i in [0, m]: 0, PP[0], ..., PP[m-1] (= Ptot)
//   QSx[i][k], i in [0, m]: QS[0] (= Qtot), ..., QS[m-1], 0
// so that PP_p(w-1) = PPx[w - lo] and QS_p(w+1) = QSx[w - lo + 1] for w in
// W_p; the local pair index of p on each interval of W_p; the column pairs'
// runs, one per column spline d, and the column pairs themselves.
size_t near_lds_bytes(int64_t ks, int64_t K)
{
    return sizeof(double) * (size_t)(2 * (ks + 1) * K + 2 * (2 * ks - 1) * (2 * ks - 1)) +
           sizeof(int) * (size_t)(kMaxOrder + 2 * kNearMaxSeg + 4);
}

__device__ __forceinline__ int pair_at(const int32_t* __restrict__ c_first, int ks, int a, int c)
{
    const int lo = (c - ks + 1) < 1 ? 1 : (c - ks + 1);
    return c_first[c] + (a - lo);
}

// FOLD: only pairs p = (a, c), a <= c, and q = (b, d), b <= d, q not before p,
// are evaluated and stored in the up to eight elements that the symmetries of
// the integral make equal (a <-> c, b <-> d, and the two electrons), so that
// every diagonal cell is read once; without it (moments from the caller's own
// containers, which need not be symmetric in a pair's splines) every column of
// the row, stored into rows (a, c) and (c, a).
//
// Bound by the latency of its gathers and the scattered stores of K
// consecutive multipoles (8 K bytes): one thread per element, the column
// pairs' indices found once per pair in LDS rather than once per element.
// Alone, FOLD against every column with a search per element: 2944 pairs x 11
// multipoles 0.038 -> 0.019 ms, 10128 x 25 0.284 -> 0.181 ms.
struct NearArgs {
    int n_pairs, n_b, n_iv, K, ks, U;
    unsigned rK;
    int n_rows;
    const PairInfo* pairs;
    const int32_t* c_first;
    const int32_t* rows;
    const double *Pw, *Qw, *PP, *QS, *Dsym;
    double* R;
};

// near workgroup blk of A.n_rows
template <bool FOLD>
__device__ __forceinline__ void near_row(const NearArgs& A, unsigned blk, double* lds)
{
    constexpr int kLanes = kNearMaxSeg;                    // one wavefront scans the runs
    const int n_pairs = A.n_pairs, n_b = A.n_b, n_iv = A.n_iv, K = A.K, ks = A.ks, U = A.U;
    const unsigned rK = A.rK;
    const PairInfo* __restrict__ pairs = A.pairs;
    const int32_t* __restrict__ c_first = A.c_first;
    const double *__restrict__ Pw = A.Pw, *__restrict__ Qw = A.Qw, *__restrict__ PP = A.PP, *__restrict__ QS = A.QS;
    const double* __restrict__ Dsym = A.Dsym;
    double* __restrict__ R = A.R;
    int4* sCol = (int4*)lds;                               // [(2 ks - 1)^2]: q, (d, b)'s pair or -1, min, max of b, d
    double* sPPx = lds + 2 * (2 * ks - 1) * (2 * ks - 1);  // [(ks+1)][K]
    double* sQSx = sPPx + (ks + 1) * K;                    // [(ks+1)][K]
    int* sUp = (int*)(sQSx + (ks + 1) * K);                // [kMaxOrder]
    int* sJ0 = sUp + kMaxOrder;                            // [kNearMaxSeg + 1]: first column pair of each spline d
    int* sB0 = sJ0 + kNearMaxSeg + 1;                      // [kNearMaxSeg]: its first b
    const int tid = threadIdx.x;
    const int p = A.rows[xcd_block(blk, A.n_rows)];         // neighbouring rows gather the same Dsym cells
    const PairInfo pp = pairs[p];
    const int lo = pp.v0, m = pp.m, hi = pp.v0 + pp.m - 1;
    const int pt = (pp.a == pp.c) ? -1 : pair_at(c_first, ks, pp.c, pp.a);   // the identical row (c, a)
    for (int e = tid; e < (ks + 1) * K; e += kThreads) {
        const int i = rK ? (int)__umulhi((unsigned)e, rK) : e, k = e - i * K;   // (e < 2^26 / K: an exact quotient)
        const size_t pb = (size_t)p * ks * K + k;
        sPPx[e] = (i == 0) ? 0.0 : PP[pb + (size_t)(i - 1) * K];
        sQSx[e] = (i >= m) ? 0.0 : QS[pb + (size_t)i * K];
    }
    if (tid < m) {
        const int vz = lo - 1 + tid;
        sUp[tid] = sym_local(pp.a - vz, pp.c - vz, ks);
    }
    // column pairs (b, d) share an interval with W_p iff max(b,d) + 2 - k <= hi
    // and min(b,d) + 1 >= lo: one run of b per d
    const int dlo = max(1, lo - 1), dhi = min(n_b, hi + ks - 2);   // dhi - dlo + 1 <= 2k - 1 <= 39
    if (tid < kLanes) {
        const int d = dlo + tid;
        int b0 = max(max(1, d - ks + 1), lo - 1);
        int b1 = FOLD ? d : min(min(d + ks - 1, n_b), hi + ks - 2);
        if (FOLD && d == pp.c) b0 = max(b0, pp.a);         // (pairs are ordered by d, then b)
        const int len = d > dhi || (FOLD && d < pp.c) ? 0 : max(0, b1 - b0 + 1);
        int inc = len;
        for (int off = 1; off < kLanes; off <<= 1) {
            const int y = __shfl_up(inc, off, kLanes);
            if (tid >= off) inc += y;
        }
        sJ0[tid] = inc - len;
        sB0[tid] = b0;
        if (tid == kLanes - 1) sJ0[kLanes] = inc;
    }
    __syncthreads();
    const int ncol = sJ0[kLanes];
    for (int j = tid; j < ncol; j += kThreads) {
        int s = 0;                       // the last run starting at or before j is the one that holds it
        for (int step = kLanes / 2; step > 0; step >>= 1)
            if (sJ0[s + step] <= j) s += step;
        const int d = dlo + s, b = sB0[s] + (j - sJ0[s]);
        sCol[j] = int4{pair_at(c_first, ks, b, d), FOLD && b != d ? pair_at(c_first, ks, d, b) : -1, min(b, d), max(b, d)};
    }
    __syncthreads();
    const int total = ncol * K;
    const int64_t rowlen = (int64_t)n_pairs * K;
    double* Rp = R + (size_t)p * rowlen;
    double* Rt = R + (size_t)(pt < 0 ? p : pt) * rowlen;
    const unsigned UK = (unsigned)(U * K);   // Dsym has n_iv*U*U*K < 2^31 entries (checked on the host)
    for (int e = tid; e < total; e += kThreads) {
        const int j = rK ? (int)__umulhi((unsigned)e, rK) : e, k = e - j * K;
        const int4 col = sCol[j];
        const int q = col.x, qt = col.y, bl = col.z, bh = col.w;
        const int v0q = max(1, bh + 2 - ks), endq = min(bl + 1, n_iv);   // q's window
        const size_t qb = (size_t)q * ks * K + k;
        double val = 0.0;
        if (v0q < lo) val = sQSx[k] * PP[qb + (size_t)(lo - 1 - v0q) * K];
        if (endq > hi) val += sPPx[m * K + k] * QS[qb + (size_t)(hi + 1 - v0q) * K];
        const int wlo = max(lo, v0q), whi = min(hi, endq);
        double acc = 0.0, dacc = 0.0;
        const double* qw = Qw + qb + (size_t)(wlo - v0q) * K;
        const double* pw = Pw + qb + (size_t)(wlo - v0q) * K;
        const double* sp = sPPx + (wlo - lo) * K + k;
        const double* sq = sQSx + (wlo - lo + 1) * K + k;
        int t = bl - (wlo - 1);                              // q's lower local spline on interval w
        unsigned Dv = (unsigned)(wlo - 1) * U * UK + (unsigned)k;
#pragma unroll 2
        for (int w = wlo; w <= whi; ++w) {
            const unsigned uq = (unsigned)(t * ks - ((t * (t - 1)) >> 1) + (bh - bl)), up = (unsigned)sUp[w - lo];
            const unsigned ulo = min(up, uq), uhi = max(up, uq);   // Dsym is read in its upper triangle
            dacc += Dsym[Dv + ulo * UK + uhi * (unsigned)K];
            acc += *qw * *sp + *pw * *sq;
            qw += K, pw += K, sp += K, sq += K, --t, Dv += U * UK;
        }
        val += acc + dacc;
        const size_t o = (size_t)q * K + k, ot = (size_t)qt * K + k;
        Rp[o] = val;
        if (pt >= 0) Rt[o] = val;
        if (FOLD) {
            const size_t op = (size_t)p * K + k, opt = (size_t)pt * K + k;
            double* const Rq = R + (size_t)q * rowlen;
            if (qt >= 0) Rp[ot] = val;
            if (qt >= 0 && pt >= 0) Rt[ot] = val;
            if (q != p) {
                Rq[op] = val;
                if (pt >= 0) Rq[opt] = val;
                if (qt >= 0) {
                    double* const Rqt = R + (size_t)qt * rowlen;
                    Rqt[op] = val;
                    if (pt >= 0) Rqt[opt] = val;
                }
            }
        }
    }
}

template <bool FOLD>
__global__ __launch_bounds__(kThreads) void k3_near(NearArgs A)
{
    extern __shared__ __align__(16) double lds[];
    near_row<FOLD>(A, blockIdx.x, lds);
}

// Far workgroups: ROWS rows x one chunk of 512 ITERS elements of rank-one
// products, two consecutive elements per thread and 16-byte store; the
// elements whose pairs' windows overlap are left to k3_near.
//
// Bound by the store of R (8 bytes per element).  What the store rate depends
// on, measured with stores alone over 20.5 GB: one 16-byte store per thread
// and row reaches 6.5-6.9 TB/s, two or four 5.5-6.5, so a workgroup takes few
// elements and lives short; and its latency has to stay short too.  Therefore
//   * no element looks at its pair: pairs are numbered column spline by
//     column spline, so the chunks right of every window of the workgroup's
//     rows, and those left of it, are told apart once per workgroup by their
//     element range, and such a chunk reads one factor table, its multipole
//     index from the offset in the chunk by a 32-bit multiplication with the
//     reciprocal of K; only the chunks near the rows' own columns (about
//     4 (2k - 1)^2 K of a row's n_pairs K elements) test every element;
//   * SHIFT: where the rows do not start on 128-byte lines (n_pairs K not a
//     multiple of 16) each row's chunks are shifted to begin on one (by up to
//     15 elements, into the chunk before), so that no line is written in
//     parts by two workgroups, which sit on different XCDs; the odd rows of an
//     odd row length take the same 16-byte stores;
//   * on the border single elements are stored without the non-temporal hint,
//     so that the parts of a line meet in L2 (0.143 -> 0.119 ms at 2944 pairs
//     x 11 multipoles; elsewhere plain stores cost 40 %).
// x_cols > 0: XCD x takes the x-th eighth of a row's chunks (x_cols of them)
// row group by row group, so that its L2 keeps that slice of the factors;
// otherwise the workgroups follow the rows.  The slices pay where the two
// factor tables take more than half of an XCD's 4 MB L2: whole builds of
// 10128 x 25 (4.1 MB) 3.27 ms in slices against 3.50 along the rows, of order
// 9 with 2.8 MB 2.29 against 2.36 and with 2.3 MB 1.50 against 1.64; of
// 6728 x 17 (1.8 MB) 1.085 against 1.042, 4444 x 17 (1.2 MB) 0.487 against
// 0.464.
// k3_far alone, 2 rows x 512 elements, against a test per element and 8-byte
// stores for odd lengths: 2944 x 11 (lines) 0.145 -> 0.119 ms; 4444 x 17
// (shifted) 0.519 -> 0.388; 3349 x 9 (odd) 0.257 -> 0.111; 10128 x 25 (lines)
// 3.18-3.60 -> 3.09.
typedef double double2_t __attribute__((ext_vector_type(2)));
typedef double double2u_t __attribute__((ext_vector_type(2), aligned(8)));   // a pair on any element boundary

constexpr int kFarLine = 16;            // elements per 128-byte line
constexpr int kFarLd = kMaxK + 2;       // a row's factors in LDS, the first one again behind the last
constexpr unsigned kFarGridY = 32768;   // row groups per grid layer
constexpr int64_t kFarSliceBytes = (int64_t)2 << 20;   // factor tables beyond which the XCDs take slices

struct FarArgs {
    int n_pairs, n_b, K, ks;
    unsigned rK, rK1;
    int far_cols, x_cols;
    const PairInfo* pairs;
    const int32_t* c_first;
    const double *Ptot, *Qtot;
    double* R;
};

// far workgroup of row group grp and chunk column bx of the launch
template <int ROWS, int ITERS, bool SHIFT>
__device__ __forceinline__ void far_chunk(const FarArgs& A, int grp, unsigned bx)
{
    constexpr int CH = 2 * kThreads * ITERS, NF = SHIFT ? ROWS : 1;
    __shared__ double sP[ROWS * kFarLd], sQ[ROWS * kFarLd];   // Ptot, Qtot of the rows
    const int n_pairs = A.n_pairs, n_b = A.n_b, K = A.K, ks = A.ks;
    const unsigned rK = A.rK, rK1 = A.rK1;
    const PairInfo* __restrict__ pairs = A.pairs;
    const int32_t* __restrict__ c_first = A.c_first;
    const double *__restrict__ Ptot = A.Ptot, *__restrict__ Qtot = A.Qtot;
    double* __restrict__ R = A.R;
    const int tid = threadIdx.x;
    const int rowlen = n_pairs * K;        // < 2^31 (checked on the host)
    const int p0 = grp * ROWS;
    if (p0 >= n_pairs) return;             // (the last grid layer can be short)
    const int nrows = (n_pairs - p0) < ROWS ? (n_pairs - p0) : ROWS;
    const int cx = A.x_cols ? (int)(bx % kXcds) * A.x_cols + (int)(bx / kXcds) : (int)bx;
    if (cx >= A.far_cols) return;          // (the last XCD's slice can be short)
    const int e0 = cx * CH;
    const unsigned uK = (unsigned)K;
    int lo[ROWS], hi[ROWS], shift[ROWS];   // uniform: scalar registers
    int lo_min = 0x7fffffff, hi_max = 0;
    double* const Rrow = R + (size_t)p0 * (size_t)rowlen;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const PairInfo pi = pairs[p0 + (r < nrows ? r : 0)];
        lo[r] = pi.v0;
        hi[r] = pi.v0 + pi.m - 1;          // last interval of the row's window
        lo_min = lo[r] < lo_min ? lo[r] : lo_min;
        hi_max = hi[r] > hi_max ? hi[r] : hi_max;
        shift[r] = SHIFT ? (int)((uintptr_t)(Rrow + (size_t)r * rowlen) / sizeof(double)) & (kFarLine - 1) : 0;
    }
    // a pair of column c has its window within [c + 2 - k, c + 1]: left of the
    // rows' windows for c <= lo_min - 2, right of them for c >= hi_max + k - 1
    const int cl = lo_min - 1 > 1 ? lo_min - 1 : 1, cr = hi_max + ks - 1 < n_b + 1 ? hi_max + ks - 1 : n_b + 1;
    const int e_left = c_first[cl] * K, e_right = c_first[cr] * K;
    const bool left = e0 + CH <= e_left, right = e0 - (SHIFT ? kFarLine - 1 : 0) >= e_right;
    // the chunk's first element is element kb - 16 K of pair qb: an element at
    // offset o + 16 K from there has pair qb - 16 + o / K and multipole o % K
    // (rK: the rounded-up reciprocal, 0 for K = 1; its quotient is exact for
    // o < 2^14, and at most one too large for e0)
    int qb = rK ? (int)__umulhi((unsigned)e0, rK) : e0;
    if (qb * K > e0) --qb;
    const unsigned kb = (unsigned)(e0 - qb * K) + kFarLine * uK;
    if ((left || right) && nrows == ROWS && e0 + CH <= rowlen && (!SHIFT || e0 > 0)) {
        // the columns' factors, and the rows' (Ptot of whichever lies left)
        const double* __restrict__ F = (left ? Ptot : Qtot) + e0;
        const double* __restrict__ G = (left ? Qtot : Ptot) + (size_t)p0 * K;
        double2u_t f[NF][ITERS];
#pragma unroll
        for (int r = 0; r < NF; ++r)
#pragma unroll
            for (int i = 0; i < ITERS; ++i) f[r][i] = *(const double2u_t*)(F - shift[r] + 2 * (i * kThreads + tid));
        for (int e = tid; e < ROWS * (K + 1); e += kThreads) {
            const int r = (int)__umulhi((unsigned)e, rK1), k = e - r * (K + 1);
            sP[r * kFarLd + k] = G[r * K + (k < K ? k : 0)];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITERS; ++i)
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const unsigned o = 2 * (i * kThreads + tid) - shift[r];
                const unsigned a = kb + o, k = rK ? a - uK * __umulhi(a, rK) : 0;
                const double* g = sP + r * kFarLd + k;
                const double2u_t v = f[SHIFT ? r : 0][i];
                __builtin_nontemporal_store(double2u_t{g[0] * v.x, g[1] * v.y},
                                            (double2u_t*)(Rrow + (size_t)r * rowlen + e0 + (int)o));
            }
        return;
    }
    for (int e = tid; e < nrows * (K + 1); e += kThreads) {
        const int r = (int)__umulhi((unsigned)e, rK1), k = e - r * (K + 1);
        const size_t g = (size_t)(p0 + r) * K + (k < K ? k : 0);
        sP[r * kFarLd + k] = Ptot[g];
        sQ[r * kFarLd + k] = Qtot[g];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITERS; ++i) {
        int e = 0;
        unsigned k = 0;
        double2u_t pt, qt;
        PairInfo a0, a1;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (SHIFT || r == 0) {   // (unshifted rows share their columns)
                const int o = 2 * (i * kThreads + tid) - shift[r];
                const unsigned a = kb + o, qo = rK ? __umulhi(a, rK) : a;
                e = e0 + o;
                k = a - qo * uK;
                const int q0 = qb - kFarLine + (int)qo, q1 = k + 1 == uK ? q0 + 1 : q0;
                // (an element before or behind the row reads a clamped place and is not stored)
                const int ec = e < 0 ? 0 : e > rowlen - 2 ? rowlen - 2 : e;
                const double2u_t pv = *(const double2u_t*)(Ptot + ec), qv = *(const double2u_t*)(Qtot + ec);
                pt = e == ec ? pv : double2u_t{pv.y, pv.x};
                qt = e == ec ? qv : double2u_t{qv.y, qv.x};
                a0 = pairs[min(max(q0, 0), n_pairs - 1)];
                a1 = pairs[min(max(q1, 0), n_pairs - 1)];
            }
            if (r >= nrows) continue;
            const bool l0 = hi[r] < a0.v0, l1 = hi[r] < a1.v0;   // the row's window lies left of the column's
            const bool f0 = e >= 0 && e < rowlen && (l0 || lo[r] > a0.v0 + a0.m - 1);
            const bool f1 = e + 1 >= 0 && e + 1 < rowlen && (l1 || lo[r] > a1.v0 + a1.m - 1);
            const double* gp = sP + r * kFarLd + k;
            const double* gq = sQ + r * kFarLd + k;
            const double2u_t v = {l0 ? gp[0] * qt.x : gq[0] * pt.x, l1 ? gp[1] * qt.y : gq[1] * pt.y};
            double* const dst = Rrow + (size_t)r * rowlen + e;
            // (an element whose windows overlap is left to k3_near)
            if (f0 && f1) *(double2u_t*)dst = v;
            else if (f0) dst[0] = v.x;
            else if (f1) dst[1] = v.y;
        }
    }
}

template <int ROWS, int ITERS, bool SHIFT>
__global__ __launch_bounds__(kThreads) void k3_far(FarArgs A)
{
    far_chunk<ROWS, ITERS, SHIFT>(A, (int)(blockIdx.z * kFarGridY + blockIdx.y), blockIdx.x);
}

// Both in one launch: the first near_y layers of workgroups take the near
// rows, the others the rank-one fill.
template <int ROWS, int ITERS, bool SHIFT, bool FOLD>
__global__ __launch_bounds__(kThreads) void k3_fill(FarArgs A, NearArgs N, unsigned near_y)
{
    extern __shared__ __align__(16) double lds[];
    const unsigned y = blockIdx.z * kFarGridY + blockIdx.y;
    if (y < near_y) {
        const unsigned blk = y * gridDim.x + blockIdx.x;
        if (blk < (unsigned)N.n_rows) near_row<FOLD>(N, blk, lds);
    } else {
        far_chunk<ROWS, ITERS, SHIFT>(A, (int)(y - near_y), blockIdx.x);
    }
}

// The store ceiling the rank-one fill is measured against: zeros over n16
// 16-byte elements, one store per thread (NT: with the non-temporal hint),
// the write pattern that reached the highest rate among those timed (more
// stores per thread, grid-stride loops and 64 contiguous bytes per thread
// were slower).
template <bool NT>
__global__ __launch_bounds__(kThreads) void k_store_fill(double2_t* __restrict__ dst, int64_t n16)
{
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n16) return;
    const double2_t z = {0.0, 0.0};
    if (NT) __builtin_nontemporal_store(z, dst + i);
    else dst[i] = z;
}

hipError_t launch_store_fill(void* dst, int64_t n16, bool nt, hipStream_t s)
{
    const unsigned grid = (unsigned)((n16 + kThreads - 1) / kThreads);
    if (nt) hipLaunchKernelGGL((k_store_fill<true>), dim3(grid), dim3(kThreads), 0, s, (double2_t*)dst, n16);
    else hipLaunchKernelGGL((k_store_fill<false>), dim3(grid), dim3(kThreads), 0, s, (double2_t*)dst, n16);
    return hipGetLastError();
}

// Dsym[v][u1][u2][k] = D[v][u1][u2][k] + D[v][u2][u1][k], in place (one
// thread per unordered local pair pair and multipole).
__global__ __launch_bounds__(256) void k_symmetrize(int n_iv, int U, int K, double* __restrict__ D)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t per_v = (int64_t)U * U * K;
    if (gid >= (int64_t)n_iv * per_v) return;
    const int v = (int)(gid / per_v);
    const int64_t rem = gid - (int64_t)v * per_v;
    const int u1 = (int)(rem / ((int64_t)U * K));
    const int u2 = (int)((rem / K) % U);
    const int k = (int)(rem % K);
    if (u2 < u1) return;
    double* a = D + (((size_t)v * U + u1) * U + u2) * K + k;
    double* b = D + (((size_t)v * U + u2) * U + u1) * K + k;
    const double s = *a + *b;
    *a = s;
    *b = s;
}

// Host: the near kernel's rows (pairs (a, c) with a <= c).
void build_near_rows(Plan& p)
{
    p.rows.clear();
    for (int64_t P = 0; P < p.n_pairs; ++P)
        if (p.pairs[P].a <= p.pairs[P].c) p.rows.push_back((int32_t)P);
}

// Host: the number of tensor elements whose pairs' windows overlap.
int64_t count_near_elements(const Plan& p)
{
    int64_t n = 0;
    const int64_t ks = p.k_s, nb = p.n_b;
    for (int64_t P = 0; P < p.n_pairs; ++P) {
        const PairInfo& pp = p.pairs[P];
        const int64_t v1p = pp.v0 + pp.m - 1;
        const int64_t cmin = std::max<int64_t>(1, pp.v0 - 1);
        const int64_t cmax = std::min<int64_t>(nb, v1p + ks - 2);
        for (int64_t Q = p.c_first[cmin]; Q < p.c_first[cmax + 1]; ++Q) {
            const PairInfo& pq = p.pairs[Q];
            if (pq.v0 <= v1p && pp.v0 <= pq.v0 + pq.m - 1) n += p.K;
        }
    }
    return n;
}

static NearArgs near_args(const Plan& p, const DevTables& d, double* R)
{
    return NearArgs{(int)p.n_pairs, (int)p.n_b, (int)p.n_iv, (int)p.K, (int)p.k_s, (int)p.U, recip32(p.K),
                    (int)p.rows.size(), d.pairs, d.c_first, d.rows, d.Pw, d.Qw, d.PP, d.QS, d.D, R};
}

hipError_t launch_tensor_near(const Plan& p, const DevTables& d, double* R, bool symmetric, hipStream_t s)
{
    if (p.rows.empty()) return hipSuccess;
    const auto kern = symmetric ? k3_near<true> : k3_near<false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)p.rows.size()), dim3(kThreads), near_lds_bytes(p.k_s, p.K), s,
                       near_args(p, d, R));
    return hipGetLastError();
}

// Shapes of the rank-one fill the autotuner chooses from: rows and groups of
// 512 elements per workgroup, and whether the rows' chunks are shifted to
// lines of memory (the shapes that take rows of odd length).
struct FarShape {
    int rows, iters;
    bool shift;
};
static constexpr FarShape kFarShapes[] = {{2, 1, false}, {2, 2, false}, {4, 1, false}, {1, 2, false},
                                          {1, 1, false}, {2, 1, true},  {2, 2, true}};

int far_variant_count() { return (int)(sizeof(kFarShapes) / sizeof(kFarShapes[0])); }

bool far_variant_valid(const Plan& p, int v)
{
    return v >= 0 && v < far_variant_count() && (kFarShapes[v].shift || (p.n_pairs * p.K) % 2 == 0);
}

// 2 rows x 512 elements, shifted unless every row starts on a line (the
// tensor does): a shifted row reads its own column factors.  Whole builds of
// 2944 pairs x 11 multipoles (lines) 0.146 ms unshifted against 0.153, of
// 10128 x 25 (lines) 3.26 against 3.24; of 4444 x 17 0.534 against 0.463.
int far_variant_default(const Plan& p) { return (p.n_pairs * p.K) % kFarLine == 0 ? 0 : 5; }

// The rank-one fill alone (near < 0), or behind the near rows in one launch
// (near: whether the moments are symmetric).
template <int V>
static void launch_far_shape(const Plan& p, const DevTables& d, double* R, int near, hipStream_t s)
{
    constexpr FarShape f = kFarShapes[V];
    const int64_t rowlen = p.n_pairs * p.K;
    // The fill reads its factors two elements at a time.  A row of one element
    // (one basis function, one multipole) has none that is rank-one: its pair
    // overlaps itself.
    const bool fill = rowlen > 1;
    if (!fill && near < 0) return;
    const int64_t per = 2 * (int64_t)kThreads * f.iters;
    // (a shifted row's last elements lie up to 15 past its last chunk)
    const unsigned cols = (unsigned)((rowlen + (f.shift ? kFarLine - 1 : 0) + per - 1) / per);
    const unsigned x_cols = 2 * sizeof(double) * rowlen > kFarSliceBytes ? (cols + kXcds - 1) / kXcds : 0;
    const unsigned gx = x_cols ? kXcds * x_cols : cols;
    const unsigned near_y = near >= 0 ? (unsigned)((p.rows.size() + gx - 1) / gx) : 0;
    const unsigned gy = (fill ? (unsigned)((p.n_pairs + f.rows - 1) / f.rows) : 0) + near_y;
    const dim3 grid(gx, std::min(gy, kFarGridY), (gy + kFarGridY - 1) / kFarGridY);
    const FarArgs a{(int)p.n_pairs, (int)p.n_b, (int)p.K, (int)p.k_s, recip32(p.K), recip32(p.K + 1), (int)cols,
                    (int)x_cols, d.pairs, d.c_first, d.Ptot, d.Qtot, R};
    if (near < 0)
        hipLaunchKernelGGL((k3_far<f.rows, f.iters, f.shift>), grid, dim3(kThreads), 0, s, a);
    else if (near > 0)
        hipLaunchKernelGGL((k3_fill<f.rows, f.iters, f.shift, true>), grid, dim3(kThreads), near_lds_bytes(p.k_s, p.K), s,
                           a, near_args(p, d, R), near_y);
    else
        hipLaunchKernelGGL((k3_fill<f.rows, f.iters, f.shift, false>), grid, dim3(kThreads), near_lds_bytes(p.k_s, p.K), s,
                           a, near_args(p, d, R), near_y);
}

static hipError_t launch_far(const Plan& p, const DevTables& d, double* R, int near, hipStream_t s)
{
    const int v = far_variant_valid(p, p.far_variant) ? p.far_variant : far_variant_default(p);
    switch (v) {
    case 0: launch_far_shape<0>(p, d, R, near, s); break;
    case 1: launch_far_shape<1>(p, d, R, near, s); break;
    case 2: launch_far_shape<2>(p, d, R, near, s); break;
    case 3: launch_far_shape<3>(p, d, R, near, s); break;
    case 4: launch_far_shape<4>(p, d, R, near, s); break;
    case 5: launch_far_shape<5>(p, d, R, near, s); break;
    default: launch_far_shape<6>(p, d, R, near, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_tensor_far(const Plan& p, const DevTables& d, double* R, hipStream_t s)
{
    return launch_far(p, d, R, -1, s);
}

hipError_t launch_tensor_fill(const Plan& p, const DevTables& d, double* R, bool symmetric, hipStream_t s)
{
    return launch_far(p, d, R, symmetric ? 1 : 0, s);
}

hipError_t launch_symmetrize(const Plan& p, const DevTables& d, hipStream_t s)
{
    const int64_t n = p.n_iv * p.U * p.U * p.K;
    hipLaunchKernelGGL(k_symmetrize, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (int)p.n_iv, (int)p.U,
                       (int)p.K, d.D);
    return hipGetLastError();
}

}  // namespace bs2e
