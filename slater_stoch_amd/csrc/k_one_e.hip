// One-electron integrals over the Gaussian fits: overlap S, nuclear
// attraction V and kinetic K of every ordered AO pair (i, k), the loop of
// src/one_e_slater.F90:87-95 over src/one_elect.F90.
//
// Each AO is the sum over its fit terms (src/one_elect.F90:20-72: i_type 1
// one term c_gauss(:,1) with the AO's powers; i_type 2 three terms
// c_gauss(:,2) with +2 on x, y or z; i_type 3 both) of its Gaussians.  Per
// primitive pair, McMurchie-Davidson with 1D Hermite coefficients E:
//   S = e^{-mu AB^2} prod_d E^{a_d b_d}_0 sqrt(pi/p), zero when
//       mu AB^2 > -ln 1e-15 (src/one_electron_sij.F90:44-46);
//   K = -1/2 of the bra Laplacian, per dimension
//       a(a-1) S(a-2) - 2 alpha (2a+1) S(a) + 4 alpha^2 S(a+2)
//       (src/one_electron_Kij.F90, with the same cut through S);
//   V = -sum_C Z_C 2pi/p e^{-mu AB^2} sum_tuv E_t E_u E_v R_tuv(p, P-C),
//       unscreened as src/NAI_pol_mult.F90 (whose own polynomial method
//       drops coefficients below 1e-9; this evaluation keeps every term).
// S, V and K are symmetric, so one workgroup takes one AO pair i >= k and
// writes both entries.  Pairs of total order up to 4 run k_one_e_pair<L>,
// where the 1D coefficients, the r^2-summed E_tuv and the R table are arrays
// of compile-time size in registers and the nuclei share one E; higher pairs
// run k_one_e with run-time orders, whose tables live in scratch memory.
// Bound: FP64 issue (Boys and R per primitive pair and nucleus).  110-AO
// random molecule, 12 nuclei: 15.3 ms with every pair on the run-time kernel,
// 0.49 ms with the five register kernels one after another, 0.40 ms side by
// side.
#include <algorithm>
#include <cmath>
#include <vector>

#include "eri_device.h"
#include "zvmc_internal.h"

using namespace zveri;

namespace {

constexpr int kOeA = 8;   // largest bra power + 2 (5G: 4 + 2; 2S, 3S: 2 + 2)
constexpr int kOeT = 13;  // largest t + 1 (bra power + 2 + ket power)
constexpr double kPi = 3.14159265358979323846;

// fit term ii of an AO of type t: coefficient set (1 or 2) and the
// coordinate that carries +2 (-1: none)
__device__ inline void fit_term(int type, int ii, int &set, int &shift)
{
    if (type == 1) {
        set = 1;
        shift = -1;
    } else if (type == 2) {
        set = 2;
        shift = ii;
    } else {
        set = ii == 0 ? 1 : 2;
        shift = ii - 1;
    }
}

// e[i][t] = E^{i,b}_t for i = 0..imax, without the e^{-mu X^2} factor
__device__ void hermite_1d(int imax, int b, double p, double xpa, double xpb,
                           double (&e)[kOeA + 1][kOeT])
{
    double cur[kOeT];
    for (int t = 0; t < kOeT; t++) cur[t] = 0.0;
    cur[0] = 1.0;
    const double h = 0.5 / p;
    for (int j = 0; j < b; j++) {
        double nxt[kOeT];
        for (int t = 0; t <= j + 1; t++)
            nxt[t] = (t > 0 ? h * cur[t - 1] : 0.0) + xpb * cur[t] + (t + 1) * cur[t + 1];
        for (int t = 0; t <= j + 1; t++) cur[t] = nxt[t];
    }
    for (int t = 0; t < kOeT; t++) e[0][t] = cur[t];
    for (int i = 0; i < imax; i++) {
        for (int t = 0; t < kOeT; t++) e[i + 1][t] = 0.0;
        for (int t = 0; t <= i + 1 + b && t < kOeT; t++)
            e[i + 1][t] = (t > 0 ? h * e[i][t - 1] : 0.0) + xpa * e[i][t] +
                          (t + 1 < kOeT ? (t + 1) * e[i][t + 1] : 0.0);
    }
}

struct OneEArgs {
    const double *center, *zeta, *c1, *c2, *g;
    const int *npower, *itype, *ngauss;
    int n, ldg, nnuc;
    const double *charge, *nuc; // nuc[3 c + d]
    double *S, *V, *K;          // column-major n x n
};

// sums over the workgroup, written to (i, k) and (k, i)
__device__ void store_sums(const OneEArgs &A, int i, int k, double s, double v, double kin)
{
    __shared__ double red[3][256];
    red[0][threadIdx.x] = s;
    red[1][threadIdx.x] = v;
    red[2][threadIdx.x] = kin;
    __syncthreads();
    for (unsigned o = blockDim.x / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o)
            for (int r = 0; r < 3; r++) red[r][threadIdx.x] += red[r][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int x = 0; x < 2; x++) {
            const size_t at = x == 0 ? (size_t)i + (size_t)k * A.n : (size_t)k + (size_t)i * A.n;
            A.S[at] = red[0][0];
            A.V[at] = red[1][0];
            A.K[at] = red[2][0];
        }
}

__global__ __launch_bounds__(256) void k_one_e(OneEArgs A, const int2 *pairs)
{
    const int i = pairs[blockIdx.x].x, k = pairs[blockIdx.x].y;
    const int ti = A.itype[i], tk = A.itype[k];
    const int nci = ti == 1 ? 1 : (ti == 2 ? 3 : 4), nck = tk == 1 ? 1 : (tk == 2 ? 3 : 4);
    const int ngi = A.ngauss[i], ngk = A.ngauss[k];
    const int nitem = ngi * ngk * nci * nck;
    const double *Ai = A.center + 3 * i, *Bk = A.center + 3 * k;
    const double thr = 34.538776394910684; // -ln(1e-15)
    double s = 0.0, v = 0.0, kin = 0.0;
    for (int w = threadIdx.x; w < nitem; w += blockDim.x) {
        const int a = w % ngi, b = (w / ngi) % ngk, ii = (w / (ngi * ngk)) % nci,
                  jj = w / (ngi * ngk * nci);
        int seti, shi, setk, shk;
        fit_term(ti, ii, seti, shi);
        fit_term(tk, jj, setk, shk);
        int pa[3], pb[3];
        for (int d = 0; d < 3; d++) {
            pa[d] = A.npower[3 * i + d] + (d == shi ? 2 : 0);
            pb[d] = A.npower[3 * k + d] + (d == shk ? 2 : 0);
        }
        const double ca = (seti == 1 ? A.c1 : A.c2)[(size_t)i * A.ldg + a];
        const double cb = (setk == 1 ? A.c1 : A.c2)[(size_t)k * A.ldg + b];
        const double dd = ca * cb;
        const double al = A.g[(size_t)i * A.ldg + a], be = A.g[(size_t)k * A.ldg + b];
        const double p = al + be, mu = al * be / p;
        double P[3], ab2 = 0.0;
        for (int d = 0; d < 3; d++) {
            P[d] = (al * Ai[d] + be * Bk[d]) / p;
            ab2 += (Ai[d] - Bk[d]) * (Ai[d] - Bk[d]);
        }
        const double arg = mu * ab2, kab = exp(-arg);
        double e[3][kOeA + 1][kOeT];
        for (int d = 0; d < 3; d++) hermite_1d(pa[d] + 2, pb[d], p, P[d] - Ai[d], P[d] - Bk[d], e[d]);
        if (!(arg > thr)) {
            const double sq = sqrt(kPi / p);
            double s1[3];
            for (int d = 0; d < 3; d++) s1[d] = e[d][pa[d]][0] * sq;
            double lap = 0.0;
            for (int d = 0; d < 3; d++) {
                const int na = pa[d];
                double d2 = -2.0 * al * (2 * na + 1) * e[d][na][0] * sq +
                            4.0 * al * al * e[d][na + 2][0] * sq;
                if (na >= 2) d2 += na * (na - 1.0) * e[d][na - 2][0] * sq;
                lap += d2 * s1[(d + 1) % 3] * s1[(d + 2) % 3];
            }
            s += dd * kab * (s1[0] * s1[1] * s1[2]);
            kin += dd * kab * (-0.5 * lap);
        }
        const int tx = pa[0] + pb[0], ty = pa[1] + pb[1], tz = pa[2] + pb[2];
        const int L = tx + ty + tz;
        double F[kOeT], R[hcount(kOeT - 1)];
        for (int c = 0; c < A.nnuc; c++) {
            const double X = P[0] - A.nuc[3 * c], Y = P[1] - A.nuc[3 * c + 1],
                         Z = P[2] - A.nuc[3 * c + 2];
            boys_rt(L, p * (X * X + Y * Y + Z * Z), F);
            hermite_R_rt(L, p, X, Y, Z, F, R);
            double acc = 0.0;
            for (int t = 0; t <= tx; t++)
                for (int u = 0; u <= ty; u++)
                    for (int q = 0; q <= tz; q++)
                        acc += e[0][pa[0]][t] * e[1][pa[1]][u] * e[2][pa[2]][q] * R[hidx(t, u, q)];
            v -= dd * A.charge[c] * (2.0 * kPi / p) * kab * acc;
        }
    }
    store_sums(A, i, k, s, v, kin);
}

// 1D Hermite coefficients of one axis for the bra powers a and a + 2 and one
// ket power b: E[0] = E^{a,b}, E[1] = E^{a+2,b} (coefficients t <= L; the
// second is used only where a + 2 + b <= L), and the overlaps E_0 at bra
// powers a - 2, a, a + 2, a + 4 in g.  All indices are compile-time
// constants.
template <int L>
__device__ __forceinline__ void hermite_axis(int a, int b, double h, double xpa, double xpb,
                                             double (&E)[2][L + 1], double (&g)[4])
{
    constexpr int N = L + 5;
    double c[N];
#pragma unroll
    for (int t = 0; t < N; t++) c[t] = t == 0 ? 1.0 : 0.0;
    auto raise = [&](double x) {
        double prev = 0.0;
#pragma unroll
        for (int t = 0; t < N; t++) {
            const double cur = c[t];
            const double up = t + 1 < N ? (t + 1) * c[t + 1] : 0.0;
            c[t] = fma(h, prev, fma(x, cur, up));
            prev = cur;
        }
    };
    g[0] = 0.0;
    for (int j = 0; j < b; j++) raise(xpb);
    for (int j = 0; j <= a + 4; j++) {
        if (j == a - 2) g[0] = c[0];
        if (j == a) {
            g[1] = c[0];
#pragma unroll
            for (int t = 0; t <= L; t++) E[0][t] = c[t];
        }
        if (j == a + 2) {
            g[2] = c[0];
#pragma unroll
            for (int t = 0; t <= L; t++) E[1][t] = c[t];
        }
        if (j == a + 4) g[3] = c[0];
        raise(xpa);
    }
}

// One AO pair of total order L (r^2 of i_type 2 included)
template <int L>
__global__ __launch_bounds__(128) void k_one_e_pair(OneEArgs A, const int2 *pairs,
                                                    const double *btab)
{
    constexpr int H = hcount(L);
    __shared__ __align__(16) double lbt[boys_words(L)];
    for (int t = threadIdx.x; t < boys_words(L); t += 128) lbt[t] = btab[boys_off(L) + t];
    __syncthreads();
    const int i = pairs[blockIdx.x].x, k = pairs[blockIdx.x].y;
    const int ngi = A.ngauss[i], ngk = A.ngauss[k];
    const double *ci = (A.itype[i] == 2 ? A.c2 : A.c1) + (size_t)i * A.ldg,
                 *ck = (A.itype[k] == 2 ? A.c2 : A.c1) + (size_t)k * A.ldg;
    const double thr = 34.538776394910684; // -ln(1e-15)
    double s = 0.0, v = 0.0, kin = 0.0;
    for (int w = threadIdx.x; w < ngi * ngk; w += 128) {
        const int ia = w % ngi, ib = w / ngi;
        const double gi = A.g[(size_t)i * A.ldg + ia], gk = A.g[(size_t)k * A.ldg + ib];
        const double dd = ci[ia] * ck[ib];
        // The bra, on which the Laplacian acts, is the primitive with the
        // smaller exponent: -2 al + 4 al^2 / 2p = -2 al be / p then cancels
        // at most one bit (with al >> be it would lose al / be).
        const bool swap = gi > gk;
        const int oa = swap ? k : i, ob = swap ? i : k;
        const double al = swap ? gk : gi, be = swap ? gi : gk;
        const bool ri = L >= 2 && A.itype[oa] == 2, rk = L >= 2 && A.itype[ob] == 2;
        const double *Ai = A.center + 3 * oa, *Bk = A.center + 3 * ob;
        int pa[3], pb[3];
        const double p = al + be, half = 0.5 / p, mu = al * be / p;
        double P[3], ab2 = 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            pa[d] = A.npower[3 * oa + d];
            pb[d] = A.npower[3 * ob + d];
            P[d] = (al * Ai[d] + be * Bk[d]) / p;
            ab2 += (Ai[d] - Bk[d]) * (Ai[d] - Bk[d]);
        }
        const double arg = mu * ab2, f = dd * exp(-arg);
        // E[axis][r^2 of k][r^2 of i]
        double E[3][2][2][L + 1], g[3][2][4];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            hermite_axis<L>(pa[d], pb[d], half, P[d] - Ai[d], P[d] - Bk[d], E[d][0], g[d][0]);
            if (rk)
                hermite_axis<L>(pa[d], pb[d] + 2, half, P[d] - Ai[d], P[d] - Bk[d], E[d][1],
                                g[d][1]);
        }
        double E3[H], lap = 0.0;
#pragma unroll
        for (int h = 0; h < H; h++) E3[h] = 0.0;
#pragma unroll
        for (int va = 0; va < (L >= 2 ? 3 : 1); va++) {
            if (va > 0 && !ri) break;
#pragma unroll
            for (int vb = 0; vb < (L >= 2 ? 3 : 1); vb++) {
                if (vb > 0 && !rk) break;
                // r^2 term on axis va of the bra and vb of the ket
                auto ax = [&](int d, int t) {
                    const bool a2 = ri && d == va, b2 = rk && d == vb;
                    const double lo = a2 ? E[d][0][1][t] : E[d][0][0][t];
                    const double hi = a2 ? E[d][1][1][t] : E[d][1][0][t];
                    return b2 ? hi : lo;
                };
                double e[3][L + 1];
#pragma unroll
                for (int d = 0; d < 3; d++)
#pragma unroll
                    for (int t = 0; t <= L; t++) e[d][t] = ax(d, t);
#pragma unroll
                for (int h = 0; h < H; h++)
                    E3[h] = fma(e[0][kH.t[h]] * e[1][kH.u[h]], e[2][kH.v[h]], E3[h]);
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const bool a2 = ri && d == va, b2 = rk && d == vb;
                    const int na = pa[d] + (a2 ? 2 : 0);
                    auto ov = [&](int q) { // overlap at bra power na - 2 + 2 q
                        const double lo = a2 ? g[d][0][q + 1] : g[d][0][q];
                        const double hi = a2 ? g[d][1][q + 1] : g[d][1][q];
                        return b2 ? hi : lo;
                    };
                    double d2 = -2.0 * al * (2 * na + 1) * ov(1) + 4.0 * al * al * ov(2);
                    if (na >= 2) d2 += na * (na - 1.0) * ov(0);
                    lap += d2 * e[(d + 1) % 3][0] * e[(d + 2) % 3][0];
                }
            }
        }
        if (!(arg > thr)) {
            const double sq = sqrt(kPi / p), s3 = f * (sq * sq * sq);
            s += s3 * E3[0];
            kin += s3 * (-0.5 * lap);
        }
        double acc = 0.0;
        for (int c = 0; c < A.nnuc; c++) {
            const double X = P[0] - A.nuc[3 * c], Y = P[1] - A.nuc[3 * c + 1],
                         Z = P[2] - A.nuc[3 * c + 2];
            double F[L + 1], R[H];
            boys_table<L>(p * (X * X + Y * Y + Z * Z), lbt, F);
            hermite_R<L>(p, X, Y, Z, F, R);
            double y[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int h = 0; h < H; h++) y[h & 3] = fma(E3[h], R[h], y[h & 3]);
            acc = fma(A.charge[c], (y[0] + y[1]) + (y[2] + y[3]), acc);
        }
        v -= f * (2.0 * kPi / p) * acc;
    }
    store_sums(A, i, k, s, v, kin);
}

template <int L>
void launch_pair(const OneEArgs &A, const int2 *pairs, int n, const double *btab, hipStream_t st)
{
    if (n > 0)
        hipLaunchKernelGGL(k_one_e_pair<L>, dim3((unsigned)n), dim3(128), 0, st, A, pairs, btab);
}

} // namespace

int zv_run_one_e(zv_context *c, int nnuc, const double *charge, const double *nuc, double *S,
                 double *V, double *K)
{
    const int n = c->n;
    for (int i = 0; i < n; i++) {
        const int deg = c->h_npower[3 * i] + c->h_npower[3 * i + 1] + c->h_npower[3 * i + 2];
        if (deg + (c->h_itype[i] != 1 ? 2 : 0) > kOeA - 2)
            return zv_fail(c, ZV_ERR_ARG, "one-electron integrals: AO %d above degree 6", i + 1);
    }
    const size_t nn = (size_t)n * n;
    // pairs i >= k by total order, those above ZV_LMAX_T last
    std::vector<int2> pairs;
    pairs.reserve(c->npair);
    int lo[ZV_LMAX_T + 3] = {};
    for (int L = 0; L <= ZV_LMAX_T + 1; L++) {
        lo[L] = (int)pairs.size();
        for (int q = 0; q < c->npair; q++)
            if (std::min(c->h_pair_L[q], ZV_LMAX_T + 1) == L)
                pairs.push_back(int2{c->h_pair_i[q] - 1, c->h_pair_k[q] - 1});
    }
    lo[ZV_LMAX_T + 2] = (int)pairs.size();
    const double *btab = nullptr;
    ZV_CHECK(zv_boys_table(c, &btab));
    ZV_CHECK(zv_ensure(c, c->b_misc, sizeof(double) * (3 * nn + 4 * (size_t)nnuc + 8) +
                                         sizeof(int2) * pairs.size()));
    double *dS = (double *)c->b_misc.p, *dV = dS + nn, *dK = dV + nn, *dq = dK + nn,
           *dnuc = dq + nnuc;
    int2 *dp = (int2 *)(dnuc + 3 * (size_t)nnuc);
    ZV_HIPCHECK(c, hipMemcpyAsync(dq, charge, sizeof(double) * nnuc, hipMemcpyHostToDevice,
                                  c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(dnuc, nuc, sizeof(double) * 3 * nnuc, hipMemcpyHostToDevice,
                                  c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(dp, pairs.data(), sizeof(int2) * pairs.size(),
                                  hipMemcpyHostToDevice, c->stream));
    // device fit arrays are padded to ZV_GMAX entries per AO
    OneEArgs a{c->d_center, c->d_zeta, c->d_c1, c->d_c2, c->d_g, c->d_npower, c->d_itype,
               c->d_ngauss, n, ZV_GMAX, nnuc, dq, dnuc, dS, dV, dK};
    {
        PhaseTimer tm(c, PH_ERI);
        // The orders write disjoint pairs, so from 256 pairs on they run side by
        // side on the context's stream and its side streams, whose other orders
        // fill the CUs that one order's last workgroups leave idle (whole call:
        // 325 pairs 250 -> 205 us, 6105 pairs 563 -> 474 us; below, the fork and
        // join cost more: 55 pairs 148 -> 158 us).  The run-time kernel stays on
        // the context's stream, whose scratch memory it needs.  The longest
        // launches come first.
        static_assert(zv_context::NSIDE >= 4, "a stream per order");
        const bool fork = pairs.size() >= 256;
        hipStream_t sts[ZV_LMAX_T + 1];
        for (int L = 0; L <= ZV_LMAX_T; L++)
            sts[L] = fork && L != 3 ? c->side[L < 3 ? L : 3] : c->stream;
        if (fork) {
            ZV_HIPCHECK(c, hipEventRecord(c->ev_fork, c->stream));
            for (int k = 0; k < 4; k++) ZV_HIPCHECK(c, hipStreamWaitEvent(c->side[k], c->ev_fork, 0));
        }
        if (lo[ZV_LMAX_T + 2] > lo[ZV_LMAX_T + 1])
            hipLaunchKernelGGL(k_one_e, dim3((unsigned)(lo[ZV_LMAX_T + 2] - lo[ZV_LMAX_T + 1])),
                               dim3(256), 0, c->stream, a, (const int2 *)dp + lo[ZV_LMAX_T + 1]);
        launch_pair<3>(a, dp + lo[3], lo[4] - lo[3], btab, sts[3]);
        launch_pair<4>(a, dp + lo[4], lo[5] - lo[4], btab, sts[4]);
        launch_pair<2>(a, dp + lo[2], lo[3] - lo[2], btab, sts[2]);
        launch_pair<1>(a, dp + lo[1], lo[2] - lo[1], btab, sts[1]);
        launch_pair<0>(a, dp + lo[0], lo[1] - lo[0], btab, sts[0]);
        ZV_HIPCHECK(c, hipGetLastError());
        if (fork)
            for (int k = 0; k < 4; k++) {
                ZV_HIPCHECK(c, hipEventRecord(c->ev_join[k], c->side[k]));
                ZV_HIPCHECK(c, hipStreamWaitEvent(c->stream, c->ev_join[k], 0));
            }
    }
    ZV_HIPCHECK(c, hipMemcpyAsync(S, dS, sizeof(double) * nn, hipMemcpyDeviceToHost, c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(V, dV, sizeof(double) * nn, hipMemcpyDeviceToHost, c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(K, dK, sizeof(double) * nn, hipMemcpyDeviceToHost, c->stream));
    ZV_HIPCHECK(c, hipStreamSynchronize(c->stream));
    return ZV_OK;
}
