// Tabulated Boys function F_n(T) = int_0^1 t^2n exp(-T t^2) dt, n = 0..L <= 8,
// of the ERI and one-electron kernels: the table, made on the host, and its
// evaluation, which also runs there (the tests compare both with the series).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

namespace zveri {

constexpr double kSqrtPi = 1.77245385090551602729816748334;

// Tabulated Boys function: polynomials in d = T - T_i about the nearest grid
// point T_i = i h, |d| <= h/2.  The Taylor series
//   F_m(T_i + d) = sum_k (-1)^k F_{m+k}(T_i) d^k / k!
// taken to k = 20 is economized (highest Chebyshev term after highest term
// dropped) to a polynomial q of degree boys_deg, within 6e-18 of F_L, on the
// host in extended precision (boys_table_host).  Three forms:
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
// of each; Taylor terms to the same error about 13 + 12.  Relative error against
// the series in extended precision: at most 9e-16 below boys_tmax, any order;
// above it every order upward adds the roundings of its factor, at most 0.3,
// 0.6, 1.0, 1.2, 1.8, 2.0, 2.5, 2.8, 3.1e-15 for L = 0..8 (15-term Taylor
// expansions on a grid of 1/2 with exp: 0.3, 0.7, 1.1, 1.5, 1.9, 2.3, 2.7, 3.2,
// 3.4e-15).
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
__device__ inline double rsqrt_estimate(double x) { return __builtin_amdgcn_rsq(x); }
__host__ inline double rsqrt_estimate(double x) { return 1.0f / sqrtf((float)x); }
__host__ __device__ inline double rsqrt_pos(double x)
{
    const double y = rsqrt_estimate(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

template <int L> __host__ __device__ inline void boys_table(double T, const double *lt, double *F)
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

// The tables of all orders (boys_off, [i][k]), in x87 extended precision.
// F_m(T) = exp(-T) sum_j (2T)^j / ((2m+1)(2m+3)...(2m+2j+1)), all terms
// positive, summed until they fall below 1e-22 of the sum, for the highest m;
// the others by the stable downward recursion.
inline std::vector<double> boys_table_host()
{
    typedef long double LD;
    constexpr int M = kBoysM, NM = kBoysLmax + M;
    // Chebyshev polynomials T_k in powers of x
    LD ch[M + 1][M + 1] = {};
    ch[0][0] = ch[1][1] = 1.0L;
    for (int k = 2; k <= M; k++)
        for (int j = 0; j <= k; j++)
            ch[k][j] = (j ? 2.0L * ch[k - 1][j - 1] : 0.0L) - ch[k - 2][j];
    std::vector<double> t((size_t)boys_off(kBoysLmax + 1));
    for (int L = 0; L <= kBoysLmax; L++)
        for (int i = 0; i < boys_cols(L); i++) {
            const LD T = (LD)i / boys_inv_h(L), delta = 0.5L / boys_inv_h(L), ex = expl(-T);
            LD F[NM + 1], term = 1.0L / (2 * NM + 1), sum = term;
            for (int j = 1; j < 2000; j++) {
                term *= 2.0L * T / (2 * NM + 2 * j + 1);
                sum += term;
                if (term < 1e-22L * sum) break;
            }
            F[NM] = sum * ex;
            for (int m = NM - 1; m >= 0; m--) F[m] = (2.0L * T * F[m + 1] + ex) / (2 * m + 1);
            // q in powers of x = d / delta
            const int D = boys_deg(L);
            LD q[M + 1], s = 1.0L;
            for (int k = 0; k <= M; k++) {
                q[k] = F[L + k] * s;
                s *= -delta / (k + 1);
            }
            for (int k = M; k > D; k--) {
                const LD a = q[k] / ch[k][k];
                for (int j = 0; j <= k; j++) q[j] -= a * ch[k][j];
            }
            double *o = t.data() + boys_off(L) + (size_t)i * boys_rows(L);
            if (boys_pair(L)) o[0] = (double)F[L - 1];
            s = 1.0L;
            for (int k = 0; k <= D; k++) {
                const LD v = q[k] * s;
                s /= delta;
                if (boys_pair(L)) o[k + 1] = (double)(-v / (k + 1));
                else o[k] = (double)v;
            }
        }
    return t;
}

} // namespace zveri
