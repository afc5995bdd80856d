// Device-side pieces shared by the ERI kernels (component and shell
// kernels): Hermite index tables, the primitive-pair layout, the Boys
// function of src/rint_sum.F90 and the McMurchie-Davidson R table.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>
#include <vector>

#include "zvmc_internal.h"

namespace zveri {

constexpr double kPi52 = 34.9868366552;
constexpr double kSqrtPi = 1.77245385090551602729816748334;

constexpr int hcount(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
// Hermite index of (t,u,v): by total s = t+u+v, then t descending, u descending
constexpr int hidx(int t, int u, int v)
{
    int s = t + u + v;
    return s * (s + 1) * (s + 2) / 6 + (s - t) * (s - t + 1) / 2 + (s - t - u);
}
struct HDecode {
    int t[969], u[969], v[969];
    constexpr HDecode() : t(), u(), v()
    {
        for (int s = 0; s <= 16; s++)
            for (int tt = s; tt >= 0; tt--)
                for (int uu = s - tt; uu >= 0; uu--) {
                    int h = hidx(tt, uu, s - tt - uu);
                    t[h] = tt;
                    u[h] = uu;
                    v[h] = s - tt - uu;
                }
    }
};
constexpr HDecode kH{};

// ------------------------------------------------------------------ pair data
struct PP {
    double *p, *ip, *Px, *Py, *Pz, *c; // [pp_total], compacted per AO pair
    double *al, *be;                   // the two exponents, same layout
    double *E;                          // [e_total]: pair P at e_off[P] + h*cap + e
    int *cnt;                           // kept entries per AO pair
    const int64_t *off, *eoff;          // per pair
    const int *cap;                     // n_gauss(i) n_gauss(k)
    const int *L;                       // Hermite order per pair
    const double *btab;                 // Boys tables of all orders (boys_table)
};

// ------------------------------------------------------------------ Boys
// F_n(T) = int_0^1 t^2n exp(-T t^2) dt for n = 0..L

// Tabulated Boys function: polynomials in d = T - T_i about the nearest grid
// point T_i = i h, |d| <= h/2.  The Taylor series
//   F_m(T_i + d) = sum_k (-1)^k F_{m+k}(T_i) d^k / k!
// taken to k = 20 is economized (highest Chebyshev term after highest term
// dropped) to a polynomial q of degree boys_deg, within 6e-18 of F_L, on the
// host in extended precision (zv_boys_table).  Three forms:
//   L = 0:      q is F_0.
//   L = 1..5:   the table holds p = F_{L-1}(T_i) - int q, whose derivative
//               is -F_L: one Horner scheme gives both, and the orders below
//               follow from F_{m-1} = (2 T F_m + exp(-T)) / (2m - 1), with
//               exp(-T) = (2L-1) F_{L-1} - 2T F_L.  That difference is as
//               accurate as each step needs (its error is an ulp of 2T F_L,
//               which the step adds to 2T F_{L-1} > 2T F_L), and the
//               exponential's 20 operations and 20 constants are saved.  From
//               boys_tmax on, where Gamma(L+1/2, T) / Gamma(L+1/2) is below
//               4e-17, F_m is the complete integral, again without exp.
//   L = 6..8:   F_L from q and the exponential, and the upward recursion with
//               it from T = 36 on: these kernels have no LDS for the longer
//               table and spend 2 % of their time here.
// A grid of h = 1/4 takes 9 + 8 multiply-adds for L = 1..4, h = 1/2 two more
// of each; Taylor terms to the same error about 13 + 12.  Relative error below
// 1.2e-15 against the series in extended precision.
// lt: the kernel's LDS copy of the table of order L, [i][k]: the coefficients
// of one expansion lie together, two to a read.
// Against the 13-term expansions, [k][i], with exp for L >= 3 and T >= 36
// (cycles per wave and 64 primitive quartets, 128-AO hydrocarbon): (0,1)
// 426 -> 339, (1,1) 666 -> 551, (1,2) 979 -> 831, (2,2) 1681 -> 1589,
// (2,3) 3288 -> 3111, of which the layout is a tenth to a third.
constexpr int kBoysLmax = 8, kBoysM = 20;
constexpr bool boys_pair(int L) { return L >= 1 && L <= 5; }
constexpr int boys_inv_h(int L) { return L <= 4 ? 4 : 2; }
constexpr int boys_deg(int L) { return L <= 4 ? 8 : 10; }
constexpr double boys_tmax(int L)
{
    constexpr double t[kBoysLmax + 1] = {36.0, 40.0, 43.5, 46.5, 49.5, 52.0, 36.0, 36.0, 36.0};
    return t[L];
}
constexpr int boys_rows(int L) { return boys_deg(L) + (boys_pair(L) ? 2 : 1); }
constexpr int boys_cols(int L) { return (int)(boys_tmax(L) * boys_inv_h(L)) + 1; }
constexpr int boys_words(int L) { return boys_rows(L) * boys_cols(L); }
constexpr int boys_off(int L) { return L == 0 ? 0 : boys_off(L - 1) + boys_words(L - 1); }

// 1/sqrt(x) for a positive normal x: the hardware estimate (about 5e-8
// relative) and one third-order step y' = y (1 + e/2 + 3 e^2/8), e = 1 - x y^2
// (remainder 5 e^3 / 16 < 1e-21), an ulp or two; it replaces a correctly
// rounded division and square root (1/s and sqrt(1/s)) in the prefactor.
__device__ inline double rsqrt_pos(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

template <int L> __device__ inline void boys_table(double T, const double *lt, double *F)
{
    constexpr int K = boys_rows(L) - 1;
    if (T < boys_tmax(L)) {
        const int i = (int)(T * boys_inv_h(L) + 0.5);
        const double d = T - (1.0 / boys_inv_h(L)) * (double)i;
        const double *c = lt + i * (K + 1);
        double b0 = c[K], b1 = 0.0;
#pragma unroll
        for (int k = K - 1; k >= 0; k--) {
            if constexpr (boys_pair(L)) b1 = k == K - 1 ? b0 : fma(b1, d, b0);
            b0 = fma(b0, d, c[k]);
        }
        if constexpr (L == 0) {
            F[0] = b0;
        } else {
            const double t2 = 2.0 * T;
            double e;
            if constexpr (boys_pair(L)) {
                F[L - 1] = b0;
                F[L] = -b1;
                e = fma(t2, b1, (2 * L - 1) * b0);
            } else {
                F[L] = b0;
                e = exp(-T);
                F[L - 1] = fma(t2, F[L], e) * (1.0 / (2 * L - 1));
            }
#pragma unroll
            for (int m = L - 2; m >= 0; m--) F[m] = fma(t2, F[m + 1], e) * (1.0 / (2 * m + 1));
        }
    } else {
        const double u_inv = rsqrt_pos(T);
        F[0] = (0.5 * u_inv) * kSqrtPi;
        if constexpr (L > 0) {
            const double tri = (0.5 * u_inv) * u_inv;
            double e = 0.0;
            if constexpr (!boys_pair(L))
                if (T <= 80.0) e = exp(-T);
#pragma unroll
            for (int m = 0; m < L; m++)
                F[m + 1] = boys_pair(L) ? F[m] * ((2 * m + 1) * tri) : (F[m] * (2 * m + 1) - e) * tri;
        }
    }
}

// Runtime order, as src/rint_sum.F90: T < 1: Taylor series of F_L and downward
// recursion; T >= 1: F_0 from erf and upward recursion, exp(-T) = 0 beyond
// T = 80.
__device__ inline void boys_rt(int L, double T, double *F)
{
    if (T < 1.0) {
        double term = 1.0, s = 1.0 / (2 * L + 1);
        for (int k = 1; k < 40; k++) {
            term = -term * T / k;
            double d = term / (2 * L + 2 * k + 1);
            s += d;
            if (fabs(d) < 1e-18) break;
        }
        F[L] = s;
        double e = exp(-T);
        for (int m = L - 1; m >= 0; m--) F[m] = (2.0 * T * F[m + 1] + e) / (2 * m + 1);
    } else {
        double u_inv = rsqrt(T);
        double u = T * u_inv;
        F[0] = ((0.5 * u_inv) * kSqrtPi) * erf(u);
        double e = T > 80.0 ? 0.0 : exp(-T);
        double tri = (0.5 * u_inv) * u_inv;
        for (int m = 0; m < L; m++) F[m + 1] = (F[m] * (2 * m + 1) - e) * tri;
    }
}

// ------------------------------------------------------------------ R table
// In place, levels n = L..0, totals s descending inside a level so that the
// level-(n+1) entries a value needs are still intact:
//   R^n_{t+1,u,v} = t R^{n+1}_{t-1,u,v} + X R^{n+1}_{t,u,v}   (same for u, v)
//   R^n_{000} = (-2 alpha)^n F_n
template <int L>
__device__ inline void hermite_R(double alpha, double X, double Y, double Z, const double *F,
                                 double *R)
{
    double m2a = -2.0 * alpha;
    double pw = 1.0;
    double pws[L + 1];
#pragma unroll
    for (int n = 0; n <= L; n++) {
        pws[n] = pw;
        pw *= m2a;
    }
#pragma unroll
    for (int n = L; n >= 0; n--) {
#pragma unroll
        for (int s = L - n; s >= 1; s--) {
#pragma unroll
            for (int t = s; t >= 0; t--) {
#pragma unroll
                for (int u = s - t; u >= 0; u--) {
                    int v = s - t - u;
                    double val;
                    if (t > 0) {
                        val = X * R[hidx(t - 1, u, v)];
                        if (t > 1) val = fma((double)(t - 1), R[hidx(t - 2, u, v)], val);
                    } else if (u > 0) {
                        val = Y * R[hidx(t, u - 1, v)];
                        if (u > 1) val = fma((double)(u - 1), R[hidx(t, u - 2, v)], val);
                    } else {
                        val = Z * R[hidx(t, u, v - 1)];
                        if (v > 1) val = fma((double)(v - 1), R[hidx(t, u, v - 2)], val);
                    }
                    R[hidx(t, u, v)] = val;
                }
            }
        }
        R[0] = pws[n] * F[n];
    }
}

__device__ inline void hermite_R_rt(int L, double alpha, double X, double Y, double Z,
                                    const double *F, double *R)
{
    double m2a = -2.0 * alpha;
    for (int n = L; n >= 0; n--) {
        for (int s = L - n; s >= 1; s--)
            for (int t = s; t >= 0; t--)
                for (int u = s - t; u >= 0; u--) {
                    int v = s - t - u;
                    double val;
                    if (t > 0) {
                        val = X * R[hidx(t - 1, u, v)];
                        if (t > 1) val += (t - 1) * R[hidx(t - 2, u, v)];
                    } else if (u > 0) {
                        val = Y * R[hidx(t, u - 1, v)];
                        if (u > 1) val += (u - 1) * R[hidx(t, u - 2, v)];
                    } else {
                        val = Z * R[hidx(t, u, v - 1)];
                        if (v > 1) val += (v - 1) * R[hidx(t, u, v - 2)];
                    }
                    R[hidx(t, u, v)] = val;
                }
        double pw = 1.0;
        for (int t = 0; t < n; t++) pw *= m2a;
        R[0] = pw * F[n];
    }
}

__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

} // namespace zveri

// ---- host side of the shell kernels (k_eri_shell.hip) ------------------
int zv_shell_ready(zv_context *c, const zveri::PP &pp);
int zv_shell_run(zv_context *c, const zveri::PP &pp, const std::vector<std::pair<int, int>> &sq,
                 DevBuf &bitem, DevBuf &bgroup, DevBuf &bpart, std::vector<char> &hplan,
                 int64_t *ngroups);
int zv_shell_scatter(zv_context *c, const DevBuf &bgroup, const DevBuf &bpart, int64_t ngroups,
                     const double *pre, double *tri);
int zv_zero(zv_context *c, double *x, int64_t n);
