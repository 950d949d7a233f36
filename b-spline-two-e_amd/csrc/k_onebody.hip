// k_onebody.hip -- one-electron matrices on the device: the overlap
// (mat_els.f90:85-118 setup_S, :330-346 compute_S) and the one-particle
// Hamiltonian of a hydrogenic potential with a complex absorbing potential
// (mat_els.f90:47-83 setup_H_one_particle, :294-321 compute_H,
// potentials.f90 V_hydrogenic, CAP_tools.f90:24-34 V_CAP).
//
//   ko_tables: one workgroup per interval, for each GL point the point
//     r = h x_q + c and weight h w_q of quad_tools.f90:29-52 and the values of
//     the k splines non-zero there, for H also their second derivatives.
//   ko_assemble: one workgroup per column j_b and group of l, one thread per
//     element of the band (i_b, j_b), |i_b - j_b| < k, and l: the reference's
//     running sum over the intervals holding both splines, in ascending order,
//     and over the GL points, in order:
//       S(i,j) += w B_i B_j
//       H(i,j) += w (-0.5 B_i B_j'' + (V_l(r) + V_CAP(r)) B_i B_j)
//     with V_l(r) = 0.5 l(l+1)/r^2 - Z/r and V_CAP(r) = -i eta (r - r_0)^order
//     for r >= r_0 (0 below).  Elements with |i_b - j_b| >= k are zero.
//
//   ko_rk_int: one thread per (k, i_b, j_b) of the RKH one-electron
//     multipoles (RKH_hamiltonian.f90:91-159 setup_r_k_int with
//     adiabatic_potentials.f90:24-34 r_k): per interval holding both splines,
//     in ascending order, the GL sum sum_q w r_k(r_q) B_i B_j, added to the
//     running total; r_k(r) = r_0^k / r^(k+1) for r > r_0 and
//     r^k / r_0^(k+1) otherwise, integer powers by squaring.
#include <algorithm>

#include "bs2e_internal.h"
#include "bspline_device.h"

namespace bs2e {

struct OneBodyArgs {
    int n_b, n_iv, ks, kgl, n_l, l_min, Z, cap_order;
    double cap_r0, eta_re, eta_im;
    double *B, *B2, *rw;       // B2 may be null (no H)
    double *S, *H;             // complex, column-major n_b x n_b (H: n_l of them); either may be null
    int group;                 // l of one workgroup
};

// Wave 0 the points and splines, wave 1 the second derivatives, side by side (a
// point a lane).
template <int KS>
__global__ __launch_bounds__(128) void ko_tables(OneBodyArgs A, const double* __restrict__ t,
                                                 const double* __restrict__ bp, const double* __restrict__ x,
                                                 const double* __restrict__ w)
{
    const int v = blockIdx.x, kgl = A.kgl, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const double lim1 = bp[v], lim2 = bp[v + 1];
    const double h = (lim2 - lim1) / 2.0, c = (lim1 + lim2) / 2.0;
    const int i1 = KS - 1 + (v + 1);
    if (wave == 0) {
        for (int q = lane; q < kgl; q += 64) {
            const double r = h * x[q] + c;
            const size_t o = (size_t)v * kgl + q;
            splines_at<KS>(t, i1, r, A.B + o * KS, 1);
            A.rw[2 * o] = r;
            A.rw[2 * o + 1] = h * w[q];
        }
    } else if (A.B2) {
        for (int q = lane; q < kgl; q += 64) {
            double d2[KS];
            splines_d2_at<KS>(t, i1, h * x[q] + c, d2);
#pragma unroll
            for (int ls = 0; ls < KS; ++ls) A.B2[((size_t)v * kgl + q) * KS + ls] = d2[ls];
        }
    }
}

// Bound by latency and, for many l, by the stores of the (mostly zero)
// matrices: the elements outside the band are stored by all threads, the band's
// are dealt out so that every lane has one, and the potential, which does not
// depend on the splines, is evaluated once per column, point and l into LDS (one
// thread per element of the whole matrix left one lane in n_b / 2k busy, each
// with the potential's divisions at every point: order 9, 400 splines, 9 l, S and
// H 211 us, now 56).
constexpr int kOneBodyL = 8;   // l of one workgroup, fewer where their potentials exceed 48 KiB of LDS

__global__ __launch_bounds__(256) void ko_assemble(OneBodyArgs A)
{
    typedef double d2_t __attribute__((ext_vector_type(2)));
    const int ks = A.ks, kgl = A.kgl, n_b = A.n_b, tid = threadIdx.x;
    extern __shared__ double lds[];
    d2_t* sV = (d2_t*)lds;             // [nl][points of the column's intervals]
    const int jb = blockIdx.x + 1, l0 = blockIdx.y * A.group;
    const int nl = A.H ? min(A.group, A.n_l - l0) : 1;
    const int iv0 = max(jb + 2 - ks, 1), npt = (min(jb + 1, A.n_iv) + 1 - iv0) * kgl;
    const size_t nn = (size_t)n_b * n_b, column = (size_t)(jb - 1) * n_b;
    d2_t* S = l0 == 0 && A.S ? (d2_t*)A.S + column : nullptr;
    d2_t* H = A.H ? (d2_t*)A.H + (size_t)l0 * nn + column : nullptr;
    for (int i = tid; i < n_b; i += 256) {
        const int d = i + 1 - jb;
        if (d < ks && -d < ks) continue;
        if (S) S[i] = d2_t{0.0, 0.0};
        if (H)
            for (int li = 0; li < nl; ++li) H[li * nn + i] = d2_t{0.0, 0.0};
    }
    if (H) {
        for (int e = tid; e < nl * npt; e += 256) {
            const int li = e / npt, l = A.l_min + l0 + li;
            const double r = A.rw[2 * ((size_t)(iv0 - 1) * kgl + e - li * npt)], cl = 0.5 * l * (l + 1);
            // V + V_CAP, V real, V_CAP = (0,-1) eta (r - r_0)^order
            double vre = cl / (r * r) - (double)A.Z / r, vim = 0.0;
            if (r >= A.cap_r0) {
                double pw = 1.0, base = r - A.cap_r0;
                for (int n = A.cap_order; n > 0; n >>= 1) {   // integer power by squaring
                    if (n & 1) pw *= base;
                    base *= base;
                }
                vre += A.eta_im * pw;    // (0,-1) (eta_re, eta_im) = (eta_im, -eta_re)
                vim = -A.eta_re * pw;
            }
            sV[e] = d2_t{vre, vim};
        }
        __syncthreads();
    }
    const int width = 2 * ks - 1;
    for (int e = tid; e < nl * width; e += 256) {
        const int li = e / width, ib = jb - ks + 1 + (e - li * width);
        if (ib < 1 || ib > n_b) continue;
        const int mx = max(ib, jb), mn = min(ib, jb);
        const int lo = max(mx + 2 - ks, 1), hi = min(mn + 1, A.n_iv);
        double s = 0.0, hr = 0.0, him = 0.0;
        for (int iv = lo; iv <= hi; ++iv) {
            const size_t o = (size_t)(iv - 1) * kgl;
            const double* bi_p = A.B + o * ks + (ib + 1 - iv);
            const double* bj_p = A.B + o * ks + (jb + 1 - iv);
            const double* rw = A.rw + 2 * o;
            if (!H) {
#pragma unroll 4
                for (int q = 0; q < kgl; ++q) s += rw[2 * q + 1] * bi_p[q * ks] * bj_p[q * ks];
                continue;
            }
            const double* d2_p = A.B2 + o * ks + (jb + 1 - iv);
            const d2_t* V = sV + li * npt + (iv - iv0) * kgl;
#pragma unroll 4
            for (int q = 0; q < kgl; ++q) {
                const double bi = bi_p[q * ks], bj = bj_p[q * ks], d2j = d2_p[q * ks], wq = rw[2 * q + 1];
                const d2_t vc = V[q];
                s += wq * bi * bj;
                hr += wq * (-0.5 * bi * d2j + vc.x * bi * bj);
                him += wq * (vc.y * bi * bj);
            }
        }
        if (S && li == 0) S[ib - 1] = d2_t{s, 0.0};
        if (H) H[li * nn + ib - 1] = d2_t{hr, him};
    }
}

__global__ __launch_bounds__(256) void ko_rk_int(int n_b, int n_iv, int ks, int kgl, int K, double r0,
                                                 const double* __restrict__ B, const double* __restrict__ rw,
                                                 double* __restrict__ out)
{
    const int64_t n = (int64_t)K * n_b * n_b;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int k = (int)(e % K);
    const int64_t ij = e / K;
    const int jb = (int)(ij / n_b) + 1, ib = (int)(ij - (int64_t)(jb - 1) * n_b) + 1;
    double acc = 0.0;
    const int d = ib > jb ? ib - jb : jb - ib;
    if (d < ks) {
        const int mx = ib > jb ? ib : jb, mn = ib < jb ? ib : jb;
        const int lo = (mx + 2 - ks) > 1 ? (mx + 2 - ks) : 1;
        const int hiv = (mn + 1) < n_iv ? (mn + 1) : n_iv;
        const double r0k = ipow_d(r0, k), r0k1 = ipow_d(r0, k + 1);
        for (int iv = lo; iv <= hiv; ++iv) {
            const int ta = ib + 1 - iv, tc = jb + 1 - iv;
            double res = 0.0;
            for (int q = 0; q < kgl; ++q) {
#pragma clang fp contract(off)
                const size_t o = (size_t)(iv - 1) * kgl + q;
                const double r = rw[2 * o], wq = rw[2 * o + 1];
                const double rk = r > r0 ? r0k / ipow_d(r, k + 1) : ipow_d(r, k) / r0k1;
                res = res + ((wq * rk) * B[o * ks + ta]) * B[o * ks + tc];   // each product rounded: no FMA
            }
            acc = acc + res;
        }
    }
    out[e] = acc;
}

template <int KS>
static void launch_tables(const OneBodyArgs& A, const DevTables& d, hipStream_t s)
{
    hipLaunchKernelGGL(ko_tables<KS>, dim3((unsigned)A.n_iv), dim3(128), 0, s, A, d.t, d.bp, d.x, d.w);
}

static hipError_t launch_tables(const OneBodyArgs& A, const DevTables& d, hipStream_t s)
{
    switch (A.ks) {
        case 2: launch_tables<2>(A, d, s); break;
        case 3: launch_tables<3>(A, d, s); break;
        case 4: launch_tables<4>(A, d, s); break;
        case 5: launch_tables<5>(A, d, s); break;
        case 6: launch_tables<6>(A, d, s); break;
        case 7: launch_tables<7>(A, d, s); break;
        case 8: launch_tables<8>(A, d, s); break;
        case 9: launch_tables<9>(A, d, s); break;
        case 10: launch_tables<10>(A, d, s); break;
        case 11: launch_tables<11>(A, d, s); break;
        case 12: launch_tables<12>(A, d, s); break;
        case 13: launch_tables<13>(A, d, s); break;
        case 14: launch_tables<14>(A, d, s); break;
        case 15: launch_tables<15>(A, d, s); break;
        case 16: launch_tables<16>(A, d, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_one_body(const Plan& p, const DevTables& d, double* B, double* B2, double* rw, int l_min, int n_l,
                           int Z, int cap_order, double cap_r0, double eta_re, double eta_im, double* S, double* H,
                           hipStream_t s)
{
    const size_t point_l = 16 * (size_t)(p.k_s * p.k_gl);   // LDS of one l
    const int group = !H ? 1 : std::max(1, std::min({kOneBodyL, n_l, (int)((48 * 1024) / point_l)}));
    const OneBodyArgs A{(int)p.n_b, (int)p.n_iv, (int)p.k_s, (int)p.k_gl, n_l, l_min, Z, cap_order, cap_r0, eta_re,
                        eta_im, B, B2, rw, S, H, group};
    const hipError_t e = launch_tables(A, d, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(ko_assemble, dim3((unsigned)p.n_b, H ? (unsigned)((n_l + group - 1) / group) : 1u), dim3(256),
                       H ? group * point_l : 0, s, A);
    return hipGetLastError();
}

hipError_t launch_rk_int(const Plan& p, const DevTables& d, double* B, double* rw, int max_k, double r0, double* out,
                         hipStream_t s)
{
    OneBodyArgs A{};
    A.n_iv = (int)p.n_iv;
    A.ks = (int)p.k_s;
    A.kgl = (int)p.k_gl;
    A.B = B;
    A.rw = rw;
    const hipError_t e = launch_tables(A, d, s);
    if (e != hipSuccess) return e;
    const int64_t n = (int64_t)(max_k + 1) * p.n_b * p.n_b;
    hipLaunchKernelGGL(ko_rk_int, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (int)p.n_b, (int)p.n_iv,
                       (int)p.k_s, (int)p.k_gl, max_k + 1, r0, B, rw, out);
    return hipGetLastError();
}

}  // namespace bs2e
