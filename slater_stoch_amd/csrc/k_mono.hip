// Exact one-centre Slater integrals on the GPU: the do_exact_monocenter
// branch of src/two_e_slater.F90:318-365 (src/compute_int_slater.F90,
// src/ijkl_slater_xnynzn.F90, src/ijkl_slater.F90, src/bigF.F90,
// src/smallg.F90, src/compute_lmin_lmax.F90, src/gaunt.F90).
//
// For four AOs x^a y^b z^c r^nsto e^{-zeta r} on one centre (a+b+c <= 2,
// as the reference's formulas require), each angular factor
// (x/r)^a (y/r)^b (z/r)^c is a short sum of complex spherical harmonics
// (Condon-Shortley phase; the table below), the radial part is r^(n-1) with
// n = 1 + a + b + c + nsto, and with the multipole expansion of 1/r12
//
//   (ik|jl) = Re sum conj(c_i) c_k conj(c_j) c_l 4 pi sum_L F_L / (2L + 1)
//             (-1)^M G(l_i L l_k; m_i -M m_k) G(l_j L l_l; m_j M m_l),
//   M = m_k - m_i = m_j - m_l,
//
// G(l1 l2 l3; m1 m2 m3) = int Y*_{l1 m1} Y_{l2 m2} Y_{l3 m3} (Gaunt, from
// Wigner 3j symbols by Racah's formula) and F_L the radial Coulomb integral
// in closed form.  The angular part depends on the two products of monomials
// x^a y^b z^c (35 of degree <= 4 each) and L only, so it is tabulated on the
// host, W_L[product ik][product jl] (49 KB), and a quartet costs at most three
// radial integrals.  One thread per one-centre quartet, which finds its AOs
// from its index in the centre's pair triangle.  Bound: latency (a few
// microseconds of dependent FP64 divisions); with the 3j symbols and the
// radial sums' factorials and powers evaluated per quartet the 37,140 quartets
// of the 110-AO random molecule took 2.04 ms, now 8 us.
#include <algorithm>
#include <cmath>
#include <map>
#include <vector>

#include "eri_device.h"
#include "zvmc_internal.h"

using zveri::hidx;

namespace {

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// (x/r)^a (y/r)^b (z/r)^c = sum_t coef_t Y_{l_t m_t}, monomials of degree
// <= 2 in the order 1, x, y, z, xx, yy, zz, xy, xz, yz
struct YTerm {
    int l, m;
    double re, im;
};
struct YExp {
    int n;
    YTerm t[4];
};
constexpr double kS4pi = 3.5449077018110318;    // sqrt(4 pi)
constexpr double kS4pi3 = 2.046653415892977;    // sqrt(4 pi / 3)
constexpr double kS2pi3 = 1.4472025091165353;   // sqrt(2 pi / 3)
constexpr double kS2pi15 = 0.6472086375185664;  // sqrt(2 pi / 15)
constexpr double kD0 = 0.5284436396808014;      // (2/3) sqrt(pi / 5)
const YExp kYExp[10] = {
    {1, {{0, 0, kS4pi, 0.0}}},
    {2, {{1, -1, kS2pi3, 0.0}, {1, 1, -kS2pi3, 0.0}}},
    {2, {{1, -1, 0.0, kS2pi3}, {1, 1, 0.0, kS2pi3}}},
    {1, {{1, 0, kS4pi3, 0.0}}},
    {4, {{0, 0, kS4pi / 3.0, 0.0}, {2, -2, kS2pi15, 0.0}, {2, 0, -kD0, 0.0}, {2, 2, kS2pi15, 0.0}}},
    {4, {{0, 0, kS4pi / 3.0, 0.0}, {2, -2, -kS2pi15, 0.0}, {2, 0, -kD0, 0.0}, {2, 2, -kS2pi15, 0.0}}},
    {2, {{0, 0, kS4pi / 3.0, 0.0}, {2, 0, 2.0 * kD0, 0.0}}},
    {2, {{2, -2, 0.0, kS2pi15}, {2, 2, 0.0, -kS2pi15}}},
    {2, {{2, -1, kS2pi15, 0.0}, {2, 1, -kS2pi15, 0.0}}},
    {2, {{2, -1, 0.0, kS2pi15}, {2, 1, 0.0, kS2pi15}}},
};

inline int monomial(int a, int b, int c)
{
    const int d = a + b + c;
    if (d == 0) return 0;
    if (d == 1) return a ? 1 : (b ? 2 : 3);
    if (a == 2) return 4;
    if (b == 2) return 5;
    if (c == 2) return 6;
    return a && b ? 7 : (a ? 8 : 9);
}

inline double fct(int n)
{
    double f = 1.0;
    for (int i = 2; i <= n; i++) f *= (double)i;
    return f;
}

// Wigner 3j symbol, Racah's formula
double w3j(int j1, int j2, int j3, int m1, int m2, int m3)
{
    if (m1 + m2 + m3 != 0 || j3 < abs(j1 - j2) || j3 > j1 + j2) return 0.0;
    if (abs(m1) > j1 || abs(m2) > j2 || abs(m3) > j3) return 0.0;
    const double tri =
        fct(j1 + j2 - j3) * fct(j1 - j2 + j3) * fct(-j1 + j2 + j3) / fct(j1 + j2 + j3 + 1);
    const double pre = sqrt(tri * fct(j1 + m1) * fct(j1 - m1) * fct(j2 + m2) * fct(j2 - m2) *
                            fct(j3 + m3) * fct(j3 - m3));
    const int kmin = std::max(0, std::max(j2 - j3 - m1, j1 - j3 + m2));
    const int kmax = std::min(j1 + j2 - j3, std::min(j1 - m1, j2 + m2));
    double s = 0.0;
    for (int k = kmin; k <= kmax; k++)
        s += ((k & 1) ? -1.0 : 1.0) /
             (fct(k) * fct(j3 - j2 + k + m1) * fct(j3 - j1 + k - m2) * fct(j1 + j2 - j3 - k) *
              fct(j1 - k - m1) * fct(j2 - k + m2));
    return ((abs(j1 - j2 - m3) & 1) ? -1.0 : 1.0) * pre * s;
}

// int dOmega Y*_{l1 m1} Y_{l2 m2} Y_{l3 m3}
double gaunt(int l1, int l2, int l3, int m1, int m2, int m3)
{
    constexpr double kInv4pi = 0.07957747154594767; // 1 / (4 pi)
    const double f = sqrt((2.0 * l1 + 1.0) * (2.0 * l2 + 1.0) * (2.0 * l3 + 1.0) * kInv4pi);
    return ((abs(m1) & 1) ? -1.0 : 1.0) * f * w3j(l1, l2, l3, 0, 0, 0) *
           w3j(l1, l2, l3, -m1, m2, m3);
}

// products of two monomials of degree <= 2, by the index of (a, b, c) in the
// order of total degree (zveri::hidx)
constexpr int kProd = 35, kLs = 5;

// W[(ik 35 + jl) 5 + L] = 4 pi / (2 L + 1) times the angular sum above
const std::vector<double> &angular_table()
{
    static const std::vector<double> tab = [] {
        // Gaunt coefficients of two factors with l <= 2
        double gt[3][5][3][5][kLs] = {};
        for (int l1 = 0; l1 < 3; l1++)
            for (int m1 = -l1; m1 <= l1; m1++)
                for (int l3 = 0; l3 < 3; l3++)
                    for (int m3 = -l3; m3 <= l3; m3++)
                        for (int L = std::abs(m1 - m3); L < kLs; L++)
                            gt[l1][m1 + 2][l3][m3 + 2][L] = gaunt(l1, L, l3, m1, m1 - m3, m3);
        // expansion of each product in (L, M): sum of conj(c_i) c_k G
        struct C {
            double re = 0.0, im = 0.0;
        };
        std::vector<C> ex((size_t)kProd * kLs * 9);
        std::vector<char> seen(kProd, 0);
        int pw[10][3];
        for (int a = 0; a <= 2; a++)
            for (int b = 0; a + b <= 2; b++)
                for (int c = 0; a + b + c <= 2; c++) {
                    int *o = pw[monomial(a, b, c)];
                    o[0] = a;
                    o[1] = b;
                    o[2] = c;
                }
        for (int i = 0; i < 10; i++)
            for (int k = 0; k < 10; k++) {
                const int p = hidx(pw[i][0] + pw[k][0], pw[i][1] + pw[k][1], pw[i][2] + pw[k][2]);
                if (seen[p]) continue;
                seen[p] = 1;
                for (int a = 0; a < kYExp[i].n; a++)
                    for (int b = 0; b < kYExp[k].n; b++) {
                        const YTerm &ti = kYExp[i].t[a], &tk = kYExp[k].t[b];
                        for (int L = 0; L < kLs; L++) {
                            const double g = gt[ti.l][ti.m + 2][tk.l][tk.m + 2][L];
                            C &o = ex[((size_t)p * kLs + L) * 9 + (tk.m - ti.m + 4)];
                            o.re += (ti.re * tk.re + ti.im * tk.im) * g;
                            o.im += (ti.re * tk.im - ti.im * tk.re) * g;
                        }
                    }
            }
        std::vector<double> t((size_t)kProd * kProd * kLs, 0.0);
        for (int p = 0; p < kProd; p++)
            for (int q = 0; q < kProd; q++)
                for (int L = 0; L < kLs; L++) {
                    double s = 0.0; // real for real AOs
                    for (int M = -L; M <= L; M++) {
                        const C &x = ex[((size_t)p * kLs + L) * 9 + M + 4];
                        const C &y = ex[((size_t)q * kLs + L) * 9 - M + 4];
                        s += ((M & 1) ? -1.0 : 1.0) * (x.re * y.re - x.im * y.im);
                    }
                    s *= 12.566370614359172 / (2.0 * L + 1.0);
                    // parity and selection rules leave rounding residues
                    t[((size_t)p * kProd + q) * kLs + L] = std::fabs(s) > 1e-15 ? s : 0.0;
                }
        return t;
    }();
    return tab;
}

// F_L = int r1^k1 e^{-g1 r1} [r1^-(L+1) int_0^r1 r2^(k2+L) e^{-g2 r2}
//                             + r1^L int_r1^inf r2^(k2-L-1) e^{-g2 r2}] dr1.
// The first term with the order of integration exchanged has the form of the
// second, and both are sums of positive terms with ratio
// (n - i) g / ((K - 1 - i) gb) from a common factor lead = (K - 1)! / g^K,
// K = k1 + k2, g = g1 + g2.
__device__ inline double radial_part(int n, int K, double ratio, double first)
{
    double t = first, s = first;
    for (int i = 0; i < n; i++) {
        t *= (double)(n - i) / (double)(K - 1 - i) * ratio;
        s += t;
    }
    return s;
}

struct MonoArgs {
    const int64_t *qoff;  // first quartet of each centre (ncent + 1)
    const int *poff;      // first pair of each centre
    const int *pairs;     // (i, k), 1-based, by pair index inside a centre
    int ncent;
    const int *npower, *nsto;
    const double *zeta, *W;
    const int64_t *kbase;
    int n;
};

__global__ __launch_bounds__(64) void k_mono_exact(int64_t nq, MonoArgs A, double *__restrict__ val,
                                                   int64_t *__restrict__ kcp)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nq) return;
    int c = 0;
    while (c + 1 < A.ncent && A.qoff[c + 1] <= t) c++;
    const int64_t r = t - A.qoff[c];
    int P = (int)((sqrt(8.0 * (double)r + 1.0) - 1.0) * 0.5);
    while ((int64_t)P * (P + 1) / 2 > r) P--;
    while ((int64_t)(P + 1) * (P + 2) / 2 <= r) P++;
    const int Q = (int)(r - (int64_t)P * (P + 1) / 2);
    const int *pp = A.pairs + 2 * (A.poff[c] + P), *pq = A.pairs + 2 * (A.poff[c] + Q);
    const int ao[4] = {pp[0], pp[1], pq[0], pq[1]};
    int prod[2], kk[2];
    double gg[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int x = ao[2 * s] - 1, y = ao[2 * s + 1] - 1;
        const int a = A.npower[3 * x] + A.npower[3 * y], b = A.npower[3 * x + 1] + A.npower[3 * y + 1],
                  d = A.npower[3 * x + 2] + A.npower[3 * y + 2];
        prod[s] = hidx(a, b, d);
        kk[s] = 2 + a + b + d + A.nsto[x] + A.nsto[y];
        gg[s] = A.zeta[x] + A.zeta[y];
    }
    const int K = kk[0] + kk[1];
    const double g = gg[0] + gg[1];
    double lead = 1.0; // (K - 1)! / g^K
    for (int i = 1; i < K; i++) lead *= (double)i / g;
    lead /= g;
    const double *W = A.W + ((size_t)prod[0] * kProd + prod[1]) * kLs;
    double sum = 0.0;
    for (int L = 0; L < kLs; L++) {
        const double w = W[L];
        if (w == 0.0 || L >= min(kk[0], kk[1])) continue;
        const double F = radial_part(kk[1] - L - 1, K, g / gg[1], lead / gg[1]) +
                         radial_part(kk[0] - L - 1, K, g / gg[0], lead / gg[0]);
        sum = fma(w, F, sum);
    }
    val[t] = sum;
    kcp[t] = zv_kcp(A.kbase, A.n, ao[0], ao[2], ao[1], ao[3]);
}

} // namespace

// One-centre quartets (all four AOs on one centre) in the reference's
// canonical orientation, replaced by their exact values; their standard
// errors set to 0 (src/two_e_slater.F90:489-493, 558-563).
int zv_run_exact_monocenter(zv_context *c, double *ijkl, double *err, int64_t *n_mono)
{
    const int n = c->n;
    // AOs grouped by centre (bitwise equal coordinates: the AOs of one atom)
    std::map<std::vector<double>, std::vector<int>> groups;
    for (int i = 1; i <= n; i++) {
        std::vector<double> key(c->h_center.begin() + 3 * (i - 1),
                                c->h_center.begin() + 3 * i);
        groups[key].push_back(i);
    }
    std::vector<int64_t> qoff(1, 0);
    std::vector<int> poff, pairs;
    for (const auto &g : groups) {
        const std::vector<int> &ao = g.second; // ascending
        for (int i : ao) {
            const int deg = c->h_npower[3 * (i - 1)] + c->h_npower[3 * (i - 1) + 1] +
                            c->h_npower[3 * (i - 1) + 2];
            if (deg > 2)
                return zv_fail(c, ZV_ERR_ARG,
                               "exact one-centre integrals: AO %d has angular degree %d; the "
                               "reference's formulas (src/ijkl_slater_xnynzn.F90) stop above d",
                               i, deg);
        }
        poff.push_back((int)pairs.size() / 2);
        for (int i : ao)
            for (int k : ao) {
                if (k > i) break;
                pairs.push_back(i);
                pairs.push_back(k);
            }
        const int64_t np = (int64_t)pairs.size() / 2 - poff.back();
        qoff.push_back(qoff.back() + np * (np + 1) / 2);
    }
    const int64_t nq = qoff.back();
    if (n_mono) *n_mono = nq;
    if (nq == 0) return ZV_OK;
    if (!c->mono_ready) {
        const std::vector<double> &w = angular_table();
        ZV_CHECK(zv_ensure(c, c->b_mono, sizeof(double) * w.size()));
        ZV_HIPCHECK(c, hipMemcpyAsync(c->b_mono.p, w.data(), sizeof(double) * w.size(),
                                      hipMemcpyHostToDevice, c->stream));
        c->mono_ready = true;
    }
    const int nc = (int)poff.size();
    ZV_CHECK(zv_ensure(c, c->b_misc, (sizeof(double) + sizeof(int64_t)) * nq +
                                         sizeof(int64_t) * qoff.size() +
                                         sizeof(int) * (poff.size() + pairs.size())));
    double *dval = (double *)c->b_misc.p;
    int64_t *dkcp = (int64_t *)(dval + nq), *dqoff = dkcp + nq;
    int *dpoff = (int *)(dqoff + nc + 1), *dpairs = dpoff + nc;
    std::vector<double> val(nq);
    std::vector<int64_t> kcp(nq);
    ZV_HIPCHECK(c, hipMemcpyAsync(dqoff, qoff.data(), sizeof(int64_t) * (nc + 1),
                                  hipMemcpyHostToDevice, c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(dpoff, poff.data(), sizeof(int) * nc, hipMemcpyHostToDevice,
                                  c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(dpairs, pairs.data(), sizeof(int) * pairs.size(),
                                  hipMemcpyHostToDevice, c->stream));
    {
        PhaseTimer tm(c, PH_ERI);
        const MonoArgs A{dqoff, dpoff, dpairs, nc, c->d_npower, c->d_nsto, c->d_zeta,
                         (const double *)c->b_mono.p, c->d_kbase, n};
        hipLaunchKernelGGL(k_mono_exact, dim3(nblk(nq, 64)), dim3(64), 0, c->stream, nq, A, dval,
                           dkcp);
        ZV_HIPCHECK(c, hipGetLastError());
    }
    ZV_HIPCHECK(c, hipMemcpyAsync(val.data(), dval, sizeof(double) * nq, hipMemcpyDeviceToHost,
                                  c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(kcp.data(), dkcp, sizeof(int64_t) * nq, hipMemcpyDeviceToHost,
                                  c->stream));
    ZV_HIPCHECK(c, hipStreamSynchronize(c->stream));
    for (int64_t t = 0; t < nq; t++) {
        if (kcp[t] < 0 || kcp[t] >= c->nint)
            return zv_fail(c, ZV_ERR_STATE, "exact one-centre integrals: bad quartet index");
        ijkl[kcp[t]] = val[t];
        if (err) err[kcp[t]] = 0.0;
    }
    return ZV_OK;
}
