// Shell-quartet analytic ERIs: the reference's gauss_ijkl
// (src/gauss_ijkl.F90:51-154) for all Cartesian components of a shell
// quartet at once, inside its Schwarz driver (src/two_e_slater.F90:230-273).
//
// The AOs of one shell (e.g. the six 3D functions of an atom) share center,
// Gaussian exponents and contraction coefficients, so all AO pairs of a
// shell pair share the primitive-pair data p, P, c_ab and the reference's
// cuts; only the Hermite coefficients E differ, and they depend on the
// primitive pair through three numbers only: 1/2p, x = beta/p and 1 - x
// (P - A = x (B - A), P - B = -(1 - x)(B - A)).  For a shell pair of order L
//
//   E^u_h(a) = sum_{n, m} G^u_{nm,h} sigma_nm(a),
//   sigma_nm = (1/2p)^n x^m (1 - x)^(L-n-m),  0 <= n <= L, 0 <= m <= L - n,
//
// with G^u fixed by the AOs' powers and B - A.  A fit of 20 Gaussians per AO
// gives up to 160,000 primitive quartets (a, c) per shell quartet, so the
// contraction over them runs first, on the sigma alone:
//
//   Z[nm, n'm', r] = sum_a sum_c w_nm(a) w'_n'm'(c) R_r(a, c) / sqrt(p + q),
//   (u|l) = C sum G^u_{nm,hu} (-1)^|hl| G^l_{n'm',hl} Z[nm, n'm', hu + hl],
//
// w = c_ab sigma / p, C the reference's 2 pi^(5/2).  Per primitive quartet
// there is one Boys evaluation, one R table and at most one multiply-add per
// (nm, r) with |r| <= n + L_l, for any number of components: a p x p | p x p
// quartet (81 integrals) costs the 35-entry R table and 105 multiply-adds.
// Powers of x and 1 - x are kept apart (every sigma of the same n has total
// degree L - n, lower degrees raised by (x + 1 - x)^k), so the expansion adds
// no cancellation to that of E itself.
//
// A wavefront owns a work item (a shell quartet or a slice of it) and runs
// 4 uniform-side times 16 lane-side primitive pairs per step: lane
// a_local * 16 + c_local.  The sum over a is v_mfma_f64_4x4x4 with R as the A
// operand (its rows the 16 c in four blocks of 4, its inner index the 4 a)
// and the weights as B (columns: 4 of the sigma), which keeps 4 sigma x 16 c
// sums in one register pair per lane; rows that need one sigma (the top
// order) take a plain multiply-add, which costs a third of the matrix
// instruction.  After the last step of a chunk of 16 c, the accumulators are
// the B operand of the same instruction with the lane weights as A, which
// sums over c; the four blocks are folded with row rotations and added to Z
// in LDS.  Z is transformed to the components once per item.
//
// Bound: FP64 issue.  The matrix instruction and FP64 vector instructions
// share the pipe (alternating them adds their times: 16.4 and 5.4 cycles), so
// the matrix form buys registers, not flops; there is no memory access in the
// loop but the next step's rows.  Before, each lane contracted R with the E of
// its components (passes of 1-4 components, Boys and R redone per pass, lane
// data reloaded per uniform pair): whole call on the 110-AO random molecule
// 402 ms, now 130 ms; on a 128-AO hydrocarbon 1190 ms, now 383 ms.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <numeric>
#include <thread>
#include <type_traits>
#include <utility>
#include <vector>

#include "eri_device.h"
#include "zvmc_internal.h"

using namespace zveri;

namespace {

// ------------------------------------------------------------------ sigma
constexpr int nsig(int L) { return (L + 1) * (L + 2) / 2; }
// sigma index s: n descending, m ascending, so that "n >= nmin" is a prefix
constexpr int sig_depth(int s)
{
    int d = 0;
    while ((d + 1) * (d + 2) / 2 <= s) d++;
    return d;
}
constexpr int sig_n(int L, int s) { return L - sig_depth(s); }
constexpr int sig_index(int L, int n, int m) { return (L - n) * (L - n + 1) / 2 + m; }
// sigmas with n >= nmin
constexpr int sig_prefix(int L, int nmin)
{
    if (nmin <= 0) return nsig(L);
    if (nmin > L) return 0;
    return (L - nmin + 1) * (L - nmin + 2) / 2;
}
constexpr int hco(int L) { return L < 0 ? 0 : hcount(L); }
constexpr int horder(int h)
{
    int s = 0;
    while (hcount(s) <= h) s++;
    return s;
}

// Row of one primitive pair: p, Px, Py, Pz, then its weights in sigma order,
// zero-padded to whole groups of four (one B operand each); an even length
// keeps rows 16-byte aligned.
constexpr int kRow[5] = {6, 8, 12, 16, 20};
constexpr int ngroup(int L) { return (nsig(L) + 3) / 4; }
// primitive pairs of a shell pair are padded with zero-weight rows to
// multiples of kLaneC, the lane-side chunk; kStepA per step on the uniform side
constexpr int kLaneC = 16, kStepA = 4;

// Expansion entries j = (sigma, h) of order L: the h with s = |h| <= n and
// k = n - s, s + 2k <= L.
constexpr int kNgMax = 98;
struct GTable {
    int n = 0;
    int sig[kNgMax] = {}, h[kNgMax] = {};
};
constexpr GTable make_gtable(int L)
{
    GTable g;
    for (int s = 0; s < nsig(L); s++) {
        const int n = sig_n(L, s);
        const int lo = 2 * n - L > 0 ? 2 * n - L : 0;
        for (int h = hco(lo - 1); h < hco(n); h++) {
            g.sig[g.n] = s;
            g.h[g.n] = h;
            g.n++;
        }
    }
    return g;
}
struct GTables {
    GTable t[5];
    constexpr GTables() : t() { for (int L = 0; L < 5; L++) t[L] = make_gtable(L); }
};
constexpr GTables kG{};
static_assert(kG.t[4].n == kNgMax, "expansion entries");

// ------------------------------------------------------------------ passes
// A class (LU, LL), LU <= LL, whose accumulators and R table do not fit in
// the registers (256 of each kind per wave) runs in passes, each a kernel of its
// own over the same primitive quartets: the rows r of order rho0..rho1 and the
// sigma groups [g0, g1).  The passes of a quartet write partial sums that the
// scatter adds.
struct Pass {
    int rho0, rho1, g0, g1;
};
constexpr int kPassMax = 4;
constexpr int npass(int LU, int LL)
{
    if (LU == 4) return 4;
    if (LU == 3 && LL == 4) return 2;
    return 1;
}
constexpr Pass pass_of(int LU, int LL, int p)
{
    const int ng = ngroup(LU);
    if (LU == 4)
        return p == 0 ? Pass{0, 5, 0, 1} : p == 1 ? Pass{0, 5, 1, 4} : p == 2 ? Pass{6, 7, 0, 4}
                                                                           : Pass{8, 8, 0, 1};
    if (LU == 3 && LL == 4) return p == 0 ? Pass{0, 7, 0, 1} : Pass{0, 5, 1, 3};
    return Pass{0, LU + LL, 0, ng};
}

// Accumulators and Z values of a pass.  A (row, group) entry with one
// needed sigma is one per-lane sum (sigma >= 0), otherwise one matrix tile.
// Needed are the sigma with n >= rho - LL (the lane side has |hl| <= LL), and
// with them the lane sigma with n' >= rho - n.
constexpr int kAccMax = 160, kZMax = 400;
struct Slots {
    int n = 0;
    int r[kAccMax] = {}, g[kAccMax] = {}, sig[kAccMax] = {}; // sig -1: matrix tile
    int z0[kAccMax] = {}, nz[kAccMax] = {};                  // Z tiles: first, count (groups g')
    int ztot = 0;
    int zslot[kZMax] = {}, zg[kZMax] = {};
};
constexpr Slots make_slots(int LU, int LL, Pass ps)
{
    Slots o;
    for (int r = hco(ps.rho0 - 1); r < hco(ps.rho1); r++) {
        const int rho = horder(r);
        const int need = sig_prefix(LU, rho - LL);
        for (int g = ps.g0; g < ps.g1; g++) {
            if (need - 4 * g <= 0) break;
            o.r[o.n] = r;
            o.g[o.n] = g;
            o.sig[o.n] = need - 4 * g == 1 ? 4 * g : -1;
            const int np = sig_prefix(LL, rho - sig_n(LU, 4 * g));
            o.z0[o.n] = o.ztot;
            o.nz[o.n] = (np + 3) / 4;
            for (int gp = 0; gp < o.nz[o.n]; gp++) {
                o.zslot[o.ztot] = o.n;
                o.zg[o.ztot] = gp;
                o.ztot++;
            }
            o.n++;
        }
    }
    return o;
}
template <int LU, int LL, int PASS> struct Cls {
    static constexpr Pass ps = pass_of(LU, LL, PASS);
    static constexpr Slots sl = make_slots(LU, LL, ps);
    static constexpr int zwords = (sl.ztot + 3) / 4 * 64; // Z tiles in LDS, 4 x 16 values a row
    // accumulators of row r: [first(r), first(r) + count(r))
    static constexpr int first(int r)
    {
        int i = 0;
        while (i < sl.n && sl.r[i] < r) i++;
        return i;
    }
    static constexpr int count(int r) { return first(r + 1) - first(r); }
};

// Position in a pass's Z area of (sigma, sigma', r), -1 if another pass has it
int z_position(int LU, const Slots &sl, int s, int sp, int r)
{
    for (int i = 0; i < sl.n; i++) {
        if (sl.r[i] != r || sl.g[i] != s / 4) continue;
        if (sp / 4 >= sl.nz[i]) return -1;
        const int z = sl.z0[i] + sp / 4;
        return z / 4 * 64 + (s & 3) + 4 * (z & 3) + 16 * (sp & 3);
    }
    return -1;
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): the hot
// loops are written out by the front end (indices are constants before any
// optimizer pass runs; left to the loop unroller the file takes ten times
// longer to compile)
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void static_for(F &&f)
{
    static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// The steps of hermite_R (eri_device.h) for order L, in place and in the same
// order: R[dst] = x_axis R[a] + coef R[b] (b -1: no second term), or, for
// axis 3, the seed R[0] = scale (-2 alpha)^n F_n with n = a.
struct RStep {
    short dst, a, b;
    signed char coef, axis;
};
template <int L> struct RProgram {
    static constexpr int N = (L + 1) * (L + 2) * (L + 3) * (L + 4) / 24;
    RStep s[N] = {};
    constexpr RProgram()
    {
        int at = 0;
        for (int n = L; n >= 0; n--) {
            for (int o = L - n; o >= 1; o--)
                for (int t = o; t >= 0; t--)
                    for (int u = o - t; u >= 0; u--) {
                        const int v = o - t - u;
                        const int ax = t > 0 ? 0 : u > 0 ? 1 : 2, k = t > 0 ? t : u > 0 ? u : v;
                        const int dt = ax == 0, du = ax == 1, dv = ax == 2;
                        RStep &e = s[at++];
                        e.dst = (short)hidx(t, u, v);
                        e.a = (short)hidx(t - dt, u - du, v - dv);
                        e.b = k > 1 ? (short)hidx(t - 2 * dt, u - 2 * du, v - 2 * dv) : (short)-1;
                        e.coef = (signed char)(k - 1);
                        e.axis = (signed char)ax;
                    }
            s[at++] = RStep{0, (short)n, -1, 0, 3};
        }
    }
};
template <int L> struct RProg {
    static constexpr RProgram<L> p{};
};

// use(r, R^0_r) is called for every row.  With FENCE it is called as the row is
// made (no later step reads it), so the table in registers is that of the
// levels above 0, the orders below L, and the compiler's scheduler is kept
// inside a level, or eight rows of the last one: left alone it starts many
// rows at once and needs 100-150 registers more.  Without, the rows are used
// after the last step, when none of them has to be waited for.
template <int L, bool FENCE, class U>
__device__ __forceinline__ void hermite_rows(double alpha, double scale, double X, double Y,
                                             double Z, const double *F, U &&use)
{
    double R[FENCE ? (L > 0 ? hcount(L - 1) : 1) : hcount(L)];
    const double m2a = -2.0 * alpha;
    double sd[L + 1];
    sd[0] = scale;
    static_for<L>([&](auto i) { sd[i + 1] = sd[i] * m2a; });
    static_for<RProgram<L>::N>([&](auto i) {
        constexpr RStep e = RProg<L>::p.s[i];
        // the last hcount(L) steps are level n = 0
        constexpr bool row = FENCE && i >= RProgram<L>::N - hcount(L);
        double v;
        if constexpr (e.axis == 3) {
            v = sd[e.a] * F[e.a];
        } else {
            const double x = e.axis == 0 ? X : e.axis == 1 ? Y : Z;
            if constexpr (e.b < 0)
                v = x * R[e.a];
            else
                v = fma((double)e.coef, R[e.b], x * R[e.a]);
        }
        if constexpr (row)
            use(std::integral_constant<int, e.dst>{}, v);
        else
            R[e.dst] = v;
        if constexpr (FENCE && (e.axis == 3 || (row && i % 8 == 0)))
            __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (!FENCE)
        static_for<hcount(L)>([&](auto r) { use(r, R[r]); });
}

struct SPD {
    const int *comp;       // AO pair index of each component
    const int *coff;       // first component of each shell pair (nsp + 1)
    const int *np;         // kept primitive pairs of each shell pair
    const int64_t *roff;   // rows of each shell pair
    const int64_t *goff;   // expansion tables of each shell pair
    const double *rows;    // [primitive pair][kRow[L]]
    const double *gu, *gl; // [component][entry]: G, and (-1)^|h| G
};

struct ShellItem {
    int su, sl;   // uniform and lane shell pair
    int s0, s1;   // steps of kStepA uniform primitive pairs
    int k0, k1;   // chunks of kLaneC lane primitive pairs
    int64_t part; // output: [ncu][ncl]
};

struct ShellGroup {
    int su, sl, ns, pad; // ns partial results [ncu][ncl] from part on
    int64_t part;
};

// Two-double arithmetic for the weights (setup only).  Z holds sums of both
// signs that cancel in the transform, so the rounding of the weights shows
// in the integrals unless every sigma of a primitive pair belongs to the
// same p and x to the last bit.
struct DD {
    double h, l;
};
__device__ inline DD dd_norm(double a, double b)
{
    const double s = a + b;
    return {s, b - (s - a)};
}
__device__ inline DD dd_mul(DD a, DD b)
{
    const double p = a.h * b.h;
    return dd_norm(p, fma(a.h, b.h, -p) + (a.h * b.l + a.l * b.h));
}
__device__ inline DD dd_one_minus(DD a)
{
    const double s = 1.0 - a.h;
    return dd_norm(s, ((1.0 - s) - a.h) - a.l);
}

// Primitive-pair rows of a shell pair (one block each)
__global__ __launch_bounds__(128) void k_pair_rows(PP pp, SPD sd, double *rows)
{
    const int s = blockIdx.x;
    const int rep = sd.comp[sd.coff[s]];
    const int L = pp.L[rep], np = sd.np[s];
    if (L > ZV_LMAX_T || np == 0) return;
    const int64_t off = pp.off[rep];
    const int rl = kRow[L], npad = (np + kLaneC - 1) / kLaneC * kLaneC;
    double *d = rows + sd.roff[s];
    for (int t = threadIdx.x; t < npad; t += blockDim.x) {
        const int64_t at = off + (t < np ? t : np - 1);
        double *o = d + (int64_t)t * rl;
        const double p = pp.p[at], ip = pp.ip[at], al = pp.al[at], be = pp.be[at];
        o[0] = p;
        o[1] = pp.Px[at];
        o[2] = pp.Py[at];
        o[3] = pp.Pz[at];
        for (int k = 4; k < rl; k++) o[k] = 0.0;
        if (t >= np) continue;
        const DD inv{ip, fma(-ip, p, 1.0) * ip}, half{0.5 * inv.h, 0.5 * inv.l};
        // x = beta / p, y = alpha / p = 1 - x, the smaller one from its exponent
        const DD sm = dd_mul(DD{al < be ? al : be, 0.0}, inv), lg = dd_one_minus(sm);
        const DD x = al < be ? lg : sm, y = al < be ? sm : lg;
        DD wn = dd_mul(DD{pp.c[at], 0.0}, inv); // c / p (1/2p)^n
        for (int n = 0; n <= L; n++) {
            for (int m = 0; m <= L - n; m++) {
                DD v = wn;
                for (int q = 0; q < m; q++) v = dd_mul(v, x);
                for (int q = 0; q < L - n - m; q++) v = dd_mul(v, y);
                o[4 + sig_index(L, n, m)] = v.h + v.l;
            }
            wn = dd_mul(wn, half);
        }
    }
}

// Expansion tables G of every component, one wavefront each.  First the 1D
// Hermite polynomials of the (up to 4) power combinations per axis,
//   e[t][k][m]: coefficient of (1/2p)^(t+k) x^m (1-x)^(a+b-t-2k-m),
// by the Hermite recursion with D = B - A along the axis, lanes over the
// coefficients; then lanes over the entries (nm, h), each summing the
// products of its order n over the three axes and the r^2 variants, with the
// degree raised from L - s - 2k to L - n by (x + 1 - x)^k.
__global__ __launch_bounds__(64) void k_expansion(PP pp, SPD sd, const int *sp_of,
                                                  const int *pair_i, const int *pair_k,
                                                  const double *center, const int *npower,
                                                  const int *itype, double *gu, double *gl)
{
    constexpr int NE = 75; // [t 5][k 3][m 5]
    __shared__ double e[2][12][NE];
    const int q = blockIdx.x, lane = threadIdx.x;
    const int P = sd.comp[q], L = pp.L[P];
    if (L > ZV_LMAX_T) return;
    const int s = sp_of[q];
    const GTable &gt = kG.t[L];
    const int64_t at = sd.goff[s] + (int64_t)(q - sd.coff[s]) * gt.n;
    const int i = pair_i[P] - 1, k = pair_k[P] - 1;
    const int ri = itype[i] == 2 ? 2 : 0, rk = itype[k] == 2 ? 2 : 0;
    // polynomial 4 axis + 2 (r^2 of i on this axis) + (r^2 of k on this axis)
    for (int t = lane; t < 12 * NE; t += 64) e[0][t / NE][t % NE] = t % NE == 0 ? 1.0 : 0.0;
    __syncthreads();
    for (int step = 0; step < 4; step++) {
        for (int x = lane; x < 12 * NE; x += 64) {
            const int pl = x / NE, c = x % NE, ax = pl / 4;
            const int t = c / 15, kk = c / 5 % 3, m = c % 5;
            const int pa = npower[3 * i + ax] + (pl & 2 ? ri : 0);
            const int pb = npower[3 * k + ax] + (pl & 1 ? rk : 0);
            const double *o = e[step & 1][pl];
            double v = o[c];
            if (step < pa + pb) {
                const double D = center[3 * k + ax] - center[3 * i + ax];
                v = t > 0 ? o[c - 15] : 0.0;
                if (step < pa) {
                    if (m > 0) v += D * o[c - 1];
                } else {
                    v -= D * o[c];
                }
                if (t < 4 && kk > 0) v += (t + 1) * o[c + 15 - 5];
            }
            e[(step + 1) & 1][pl][c] = v;
        }
        __syncthreads();
    }
    const int vi = ri ? 3 : 1, vk = rk ? 3 : 1;
    for (int j = lane; j < gt.n; j += 64) {
        const int sg = gt.sig[j], h = gt.h[j], t = kH.t[h], u = kH.u[h], v = kH.v[h];
        const int dp = sig_depth(sg), n = L - dp, M = sg - dp * (dp + 1) / 2;
        const int kk = n - (t + u + v);
        double acc = 0.0;
        for (int w = 0; w < vi * vk; w++) {
            const int a = w / vk, b = w % vk;
            const double *E[3];
            int d[3];
            for (int ax = 0; ax < 3; ax++) {
                const int xi = ri && a == ax, xk = rk && b == ax;
                E[ax] = e[0][4 * ax + 2 * xi + xk];
                d[ax] = npower[3 * i + ax] + npower[3 * k + ax] + (xi ? 2 : 0) + (xk ? 2 : 0);
            }
            for (int kx = 0; kx <= kk && t + 2 * kx <= d[0]; kx++)
                for (int ky = 0; kx + ky <= kk && u + 2 * ky <= d[1]; ky++) {
                    const int kz = kk - kx - ky;
                    if (v + 2 * kz > d[2]) continue;
                    const double *ex = E[0] + 15 * t + 5 * kx, *ey = E[1] + 15 * u + 5 * ky,
                                 *ez = E[2] + 15 * v + 5 * kz;
                    for (int mx = 0; mx <= d[0] - t - 2 * kx; mx++)
                        for (int my = 0; my <= d[1] - u - 2 * ky; my++) {
                            const double xy = ex[mx] * ey[my];
                            double bin = 1.0; // binomial(kk, z)
                            for (int z = 0; z <= kk; z++) {
                                const int mz = M - mx - my - z;
                                if (mz >= 0 && mz <= d[2] - v - 2 * kz) acc += bin * xy * ez[mz];
                                bin = bin * (kk - z) / (z + 1);
                            }
                        }
                }
        }
        gu[at + j] = acc;
        gl[at + j] = (t + u + v) & 1 ? -acc : acc;
    }
}

// Sums over the four blocks of 4 lanes in each row of 16: the partner 8 and 4
// lanes away (row rotation by 8; shifts by 4 either way, merged by bank).
__device__ __forceinline__ double lane_xor8(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x128, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x128, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ int lane_xor4(int v)
{
    const int up = __builtin_amdgcn_update_dpp(0, v, 0x104, 0xf, 0x5, false); // lane + 4
    return __builtin_amdgcn_update_dpp(up, v, 0x114, 0xf, 0xa, false);        // lane - 4
}
__device__ __forceinline__ double lane_xor4(double v)
{
    const long long b = __double_as_longlong(v);
    return __longlong_as_double(((long long)lane_xor4((int)(b >> 32)) << 32) |
                                (unsigned)lane_xor4((int)b));
}

// One wave's LDS accesses are in order; this keeps the compiler from moving
// them across.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// uniform components transformed at a time: those of the largest shell pair
// (p x s, p x p, p x d) or as many as nine
constexpr int transform_rows(int LU) { return LU == 0 ? 1 : LU == 1 ? 3 : 9; }

// Estimated registers (accumulators, R table, the rest) and LDS doubles of one
// wave of a class's pass
constexpr int quartet_regs(int LU, int LL, int p, bool fence)
{
    const Pass ps = pass_of(LU, LL, p);
    return 2 * (make_slots(LU, LL, ps).n + hco(fence ? ps.rho1 - 1 : ps.rho1)) + 60;
}
constexpr int quartet_lds(int LU, int LL, int p)
{
    return (make_slots(LU, LL, pass_of(LU, LL, p)).ztot + 3) / 4 * 64 + 1 +
           transform_rows(LU) * kG.t[LL].n;
}
// Waves per SIMD a pass is compiled for: two, in workgroups of four waves that
// share the Boys table, where registers and LDS (two workgroups per CU) allow
// it; otherwise one, each wave a workgroup of its own, whose transform reuses
// the table's LDS (four per CU need 40 KB each).
constexpr int quartet_waves(int LU, int LL, int p)
{
    return quartet_regs(LU, LL, p, true) <= 250 &&
                   (4 * quartet_lds(LU, LL, p) + boys_words(pass_of(LU, LL, p).rho1)) * 8 <=
                       81920
               ? 2
               : 1;
}
constexpr int quartet_wpb(int LU, int LL, int p) { return quartet_waves(LU, LL, p) >= 2 ? 4 : 1; }
// instances that would leave their register budget (256 or 512) without:
// fences cost the others 3-7 % ((2, 2) and (2, 3) on the 128-AO hydrocarbon)
constexpr bool quartet_fence(int LU, int LL, int p)
{
    return quartet_regs(LU, LL, p, false) > (quartet_waves(LU, LL, p) >= 2 ? 230 : 400);
}

template <int LU, int LL, int PASS>
__global__ __launch_bounds__(64 * quartet_wpb(LU, LL, PASS))
__attribute__((amdgpu_waves_per_eu(quartet_waves(LU, LL, PASS)))) void
k_eri_quartet(SPD sd, const ShellItem *__restrict__ items, int nitems,
              const double *__restrict__ btab, const short *__restrict__ ztab,
              const double *__restrict__ rows, const double *__restrict__ gu,
              const double *__restrict__ gl, double *__restrict__ part)
{
    using C = Cls<LU, LL, PASS>;
    constexpr int WPB = quartet_wpb(LU, LL, PASS);
    constexpr int L = C::ps.rho1, NS = C::sl.n, NZ = C::sl.ztot;
    constexpr int RU = kRow[LU], RLn = kRow[LL], GU = ngroup(LU), GL = ngroup(LL);
    constexpr int NGU = kG.t[LU].n, NGL = kG.t[LL].n, TR = transform_rows(LU);
    constexpr bool OWN = WPB > 1; // transform rows beside the table, not in its place
    constexpr int NT = TR * NGL;
    __shared__ __align__(16) double lbt[OWN || boys_words(L) > NT ? boys_words(L) : NT];
    __shared__ double zall[WPB][C::zwords + 1]; // the last word stays 0
    __shared__ double tall[OWN ? WPB * NT : 1];
    for (int t = threadIdx.x; t < boys_words(L); t += 64 * WPB) lbt[t] = btab[boys_off(L) + t];
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int ii = blockIdx.x * WPB + wave;
    if (ii >= nitems) return;
    const ShellItem it = items[ii];
    double *Z = zall[wave];
    for (int t = lane; t < C::zwords + 1; t += 64) Z[t] = 0.0;
    const int al = lane >> 4, cl = lane & 15, j4 = lane & 3;
    const double *ub = rows + sd.roff[it.su] + al * RU;
    const double *lb = rows + sd.roff[it.sl];
    const bool b1 = (lane & 4) != 0, b2 = (lane & 8) != 0; // block of 4 lanes in its row of 16

    for (int k = it.k0; k < it.k1; k++) {
        const double *lr = lb + (int64_t)(kLaneC * k + cl) * RLn;
        const double q = lr[0], Qx = lr[1], Qy = lr[2], Qz = lr[3];
        // lane weights as the A operand of the sum over c: row 4 g' + j4,
        // inner index c = 4 block + lane / 16
        const double *lw = lb + (int64_t)(kLaneC * k + (lane >> 2 & 3) * 4 + al) * RLn + 4 + j4;
        double Wl[GL];
#pragma unroll
        for (int g = 0; g < GL; g++) Wl[g] = 4 * g + 4 <= RLn - 4 || 4 * g + j4 < RLn - 4 ? lw[4 * g] : 0.0;
        double V[NS];
#pragma unroll
        for (int i = 0; i < NS; i++) V[i] = 0.0;
        // uniform rows one step ahead
        double np_, nx, ny, nz, nw[GU], ns0;
        auto load_u = [&](int s) {
            const double *r = ub + (int64_t)(kStepA * s) * RU;
            np_ = r[0];
            nx = r[1];
            ny = r[2];
            nz = r[3];
            ns0 = r[4];
            if constexpr (LU > 0) {
#pragma unroll
                for (int g = C::ps.g0; g < C::ps.g1; g++) nw[g] = r[4 + 4 * g + j4];
            }
        };
        load_u(it.s0);
        for (int s = it.s0; s < it.s1; s++) {
            const double p = np_, X = nx - Qx, Y = ny - Qy, Zc = nz - Qz, w0 = ns0;
            double w[GU];
#pragma unroll
            for (int g = C::ps.g0; g < C::ps.g1; g++) w[g] = LU > 0 ? nw[g] : 0.0;
            if (s + 1 < it.s1) load_u(s + 1);
            const double sum = p + q;
            const double rs = rsqrt_pos(sum);
            const double alpha = (p * q) * (rs * rs);
            const double T = alpha * fma(X, X, fma(Y, Y, Zc * Zc));
            double F[L + 1];
            boys_table<L>(T, lbt, F);
            hermite_rows<L, quartet_fence(LU, LL, PASS)>(alpha, rs, X, Y, Zc, F, [&](auto rc, double v) {
                constexpr int r = decltype(rc)::value;
                static_for<C::count(r)>([&](auto k) {
                    constexpr int i = C::first(r) + k;
                    if constexpr (C::sl.sig[i] >= 0)
                        V[i] = fma(v, w0, V[i]);
                    else
                        V[i] = __builtin_amdgcn_mfma_f64_4x4x4f64(v, w[C::sl.g[i]], V[i], 0, 0, 0);
                });
            });
        }
        // per-lane sums (one of the 4 a each) to tile form: summed over a
        const double hot = j4 == 0 ? 1.0 : 0.0;
        static_for<NS>([&](auto i) {
            if constexpr (C::sl.sig[i] >= 0)
                V[i] = __builtin_amdgcn_mfma_f64_4x4x4f64(V[i], hot, 0.0, 0, 0, 0);
        });
        // Z tiles, four at a time: sum over c, then over the blocks, block b
        // keeping tile b
        static_for<(NZ + 3) / 4>([&](auto zq) {
            double t4[4];
            static_for<4>([&](auto b) {
                constexpr int z = 4 * zq + b;
                if constexpr (z < NZ)
                    t4[b] = __builtin_amdgcn_mfma_f64_4x4x4f64(Wl[C::sl.zg[z]],
                                                               V[C::sl.zslot[z]], 0.0, 0, 0, 0);
                else
                    t4[b] = 0.0;
            });
            const double y0 = (b2 ? t4[2] : t4[0]) + lane_xor8(b2 ? t4[0] : t4[2]);
            const double y1 = (b2 ? t4[3] : t4[1]) + lane_xor8(b2 ? t4[1] : t4[3]);
            Z[zq * 64 + lane] += (b1 ? y1 : y0) + lane_xor4(b1 ? y0 : y1);
        });
    }
    wave_lds_fence();
    // transform to the components
    double *T = OWN ? tall + wave * NT : lbt;
    const int cu0 = sd.coff[it.su], ncu = sd.coff[it.su + 1] - cu0;
    const int ncl = sd.coff[it.sl + 1] - sd.coff[it.sl];
    const double *Gu = gu + sd.goff[it.su], *Gl = gl + sd.goff[it.sl];
    for (int u0 = 0; u0 < ncu; u0 += TR) {
        const int nu = ncu - u0 < TR ? ncu - u0 : TR;
        for (int t = lane; t < nu * NGL; t += 64) {
            const int u = t / NGL, jl = t - u * NGL;
            const double *g = Gu + (int64_t)(u0 + u) * NGU;
            const short *zp = ztab + jl;
            double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 14
            for (int j = 0; j < NGU; j++) v[j & 3] = fma(g[j], Z[zp[j * NGL]], v[j & 3]);
            T[t] = (v[0] + v[1]) + (v[2] + v[3]);
        }
        wave_lds_fence();
        for (int t = lane; t < nu * ncl; t += 64) {
            const int u = t / ncl, l = t - u * ncl;
            const double *g = Gl + (int64_t)l * NGL;
            double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 14
            for (int j = 0; j < NGL; j++) v[j & 3] = fma(g[j], T[u * NGL + j], v[j & 3]);
            part[it.part + (int64_t)u0 * ncl + t] = kPi52 * ((v[0] + v[1]) + (v[2] + v[3]));
        }
        wave_lds_fence();
    }
}

// Sum the slices of each group and write triangle order.  A diagonal shell
// quartet (su == sl) holds every component quartet twice; the (P >= Q) copy
// is written.  With pre, off-diagonal component quartets failing
// |pre_P pre_Q| >= 1e-30 are written as zero (src/two_e_slater.F90:268-272).
// A small molecule's quartets are cut into thousands of slices of one or a
// few components, so the workgroup's threads share the slices of each
// component (fixed shares, added in a fixed order): with one thread adding
// them all, this kernel took more than half of a 7-AO molecule's time and the
// long sequential sum was its largest rounding error.
__global__ __launch_bounds__(256) void k_shell_scatter(const ShellGroup *groups, SPD sd,
                                                       const double *part, const double *pre,
                                                       double *tri)
{
    __shared__ double red[256];
    const ShellGroup g = groups[blockIdx.x];
    const int bu = sd.coff[g.su], bl = sd.coff[g.sl];
    const int nl = sd.coff[g.sl + 1] - bl, n = (sd.coff[g.su + 1] - bu) * nl;
    const int width = n < 256 ? n : 256, team = min(256 / width, g.ns);
    const int tc = threadIdx.x % width, ts = threadIdx.x / width;
    for (int t0 = 0; t0 < n; t0 += width) {
        const int t = t0 + tc;
        const bool mine = ts < team && t < n;
        double v = 0.0;
        if (mine) {
            const double *p = part + g.part + t;
            double a[4] = {0.0, 0.0, 0.0, 0.0};
            int s = ts;
            for (; s + 3 * team < g.ns; s += 4 * team)
#pragma unroll
                for (int k = 0; k < 4; k++) a[k] += p[(int64_t)(s + k * team) * n];
            for (; s < g.ns; s += team) a[0] += p[(int64_t)s * n];
            v = (a[0] + a[1]) + (a[2] + a[3]);
        }
        if (team > 1) {
            __syncthreads();
            red[threadIdx.x] = v;
            __syncthreads();
            for (int h = 1; h < team; h <<= 1) {
                double w = 0.0;
                const bool add = mine && ts % (2 * h) == 0 && ts + h < team;
                if (add) w = red[threadIdx.x + h * width];
                if (add) red[threadIdx.x] = v += w;
                __syncthreads();
            }
        }
        if (!mine || ts > 0) continue;
        const int u = t / nl, l = t - u * nl;
        const int P = sd.comp[bu + u], Q = sd.comp[bl + l];
        if (g.su == g.sl && P < Q) continue;
        if (pre && P != Q && fabs(pre[P] * pre[Q]) < 1.0e-30) v = 0.0;
        tri[P > Q ? zv_tri(P, Q) : zv_tri(Q, P)] = v;
    }
}

__global__ void k_zero(double *x, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0.0;
}

// ------------------------------------------------------------------ launches
// bucket b = 25 (2 pass) + 5 LU + LL: the statistics slot is 36 + b
constexpr int kNB = 25 * 2 * kPassMax;
constexpr int bucket_of(int LU, int LL, int pass) { return 50 * pass + 5 * LU + LL; }

struct LaunchArgs {
    SPD sd;
    const ShellItem *items;
    int n;
    const double *btab;
    const short *ztab;
    double *part;
    hipStream_t st;
};

template <int LU, int LL, int PASS> void launch_quartet(const LaunchArgs &a)
{
    constexpr int WPB = quartet_wpb(LU, LL, PASS), most = (int)(kLaunchThreads / 64);
    for (int i = 0, n; i < a.n; i += n) {
        n = std::min(a.n - i, most);
        hipLaunchKernelGGL((k_eri_quartet<LU, LL, PASS>), dim3((unsigned)((n + WPB - 1) / WPB)),
                           dim3(64 * WPB), 0, a.st, a.sd, a.items + i, n, a.btab, a.ztab,
                           a.sd.rows, a.sd.gu, a.sd.gl, a.part);
    }
}

struct ClassInfo {
    void (*launch)(const LaunchArgs &) = nullptr;
    double step = 0.0, chunk = 0.0; // estimated cycles per step and per chunk
    double acc = 0.0;               // multiply-adds per primitive quartet
    std::vector<short> ztab;
};

// Estimated SIMD cycles at two waves per SIMD: 5.5 per FP64 vector
// instruction, 16.4 per 4x4x4 matrix instruction (both measured on MI355X).
template <int LU, int LL, int PASS> void add_class(ClassInfo *t)
{
    using C = Cls<LU, LL, PASS>;
    ClassInfo &c = t[bucket_of(LU, LL, PASS)];
    c.launch = launch_quartet<LU, LL, PASS>;
    const int L = C::ps.rho1;
    int ns = 0, nm = 0;
    for (int i = 0; i < C::sl.n; i++) (C::sl.sig[i] >= 0 ? ns : nm)++;
    const double r = (L + 1) * (L + 2) * (L + 3) * (L + 4) / 24.0 - (L + 1);
    c.step = 5.5 * (62.0 + 3.0 * L + 1.7 * r + ns) + 16.4 * nm;
    c.chunk = 1500.0 + 16.4 * (ns + C::sl.ztot) + 30.0 * C::sl.ztot;
    for (int i = 0; i < C::sl.n; i++) {
        const int need = sig_prefix(LU, horder(C::sl.r[i]) - LL) - 4 * C::sl.g[i];
        c.acc += need < 4 ? need : 4;
    }
    const GTable &u = kG.t[LU], &l = kG.t[LL];
    c.ztab.assign((size_t)u.n * l.n, (short)C::zwords);
    for (int j = 0; j < u.n; j++)
        for (int jl = 0; jl < l.n; jl++) {
            const int hu = u.h[j], hl = l.h[jl];
            const int r3 = hidx(kH.t[hu] + kH.t[hl], kH.u[hu] + kH.u[hl], kH.v[hu] + kH.v[hl]);
            const int z = z_position(LU, C::sl, u.sig[j], l.sig[jl], r3);
            if (z >= 0) c.ztab[(size_t)j * l.n + jl] = (short)z;
        }
    if constexpr (PASS + 1 < npass(LU, LL)) add_class<LU, LL, PASS + 1>(t);
}

const ClassInfo *class_table()
{
    static ClassInfo *t = [] {
        static ClassInfo tab[kNB];
        add_class<0, 0, 0>(tab);
        add_class<0, 1, 0>(tab);
        add_class<0, 2, 0>(tab);
        add_class<0, 3, 0>(tab);
        add_class<0, 4, 0>(tab);
        add_class<1, 1, 0>(tab);
        add_class<1, 2, 0>(tab);
        add_class<1, 3, 0>(tab);
        add_class<1, 4, 0>(tab);
        add_class<2, 2, 0>(tab);
        add_class<2, 3, 0>(tab);
        add_class<2, 4, 0>(tab);
        add_class<3, 3, 0>(tab);
        add_class<3, 4, 0>(tab);
        add_class<4, 4, 0>(tab);
        return tab;
    }();
    return t;
}

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// Boys values, R recursion (2 FMA per entry over all levels) and prefactor
double boys_r_flops(int L)
{
    double HR4 = (L + 1) * (L + 2) * (L + 3) * (L + 4) / 24.0;
    return 25.0 + 3.0 * (L + 1) + 4.0 * (HR4 - 1.0) + 12.0;
}

// ------------------------------------------------------------------ planner
// A plan's items (bucket b at [lo[b], lo[b + 1])) and groups live in the
// caller's host buffer (items, then groups), from which they are copied to
// the device as they are.
struct Plan {
    ShellItem *items = nullptr;
    size_t nitems = 0;
    int lo[kNB + 1] = {};
    ShellGroup *groups = nullptr;
    size_t ngroups = 0;
    int64_t npart = 0;
    double units[kNB] = {}, flops[kNB] = {}; // per bucket
    double host_ms[4] = {};                  // orientation, items, join, bucket sort
};

inline int nchunk(int np) { return (np + kLaneC - 1) / kLaneC; }
inline int nstep(int np) { return (np + kStepA - 1) / kStepA; }

// Estimated cycles of one pass over a shell quartet and of its transform to
// the components.
double quartet_cost(const ClassInfo &ci, int npu, int npl)
{
    return nchunk(npl) * (nstep(npu) * ci.step + ci.chunk);
}
double transform_cost(int LU, int LL, int ncu, int ncl)
{
    const double gu = kG.t[LU].n, gl = kG.t[LL].n;
    return 2500.0 + 12.0 * (ncu * gl * gu + (double)ncu * ncl * gl) / 64.0;
}

// Host threads for the planner: up to 16 (the host share of one GPU), one
// for short lists.
int plan_threads(size_t n)
{
    if (n < 20000) return 1;
    const unsigned hw = std::thread::hardware_concurrency();
    return (int)std::max(1u, std::min(16u, hw ? hw : 1u));
}

// run f(t) for t = 0 .. nt-1, on nt - 1 extra threads and this one; a
// range whose thread cannot be started runs here (f(t) are independent)
template <typename F> void run_threads(int nt, F &&f)
{
    std::vector<std::thread> th;
    int started = 1;
    for (int t = 1; t < nt; t++, started++) {
        try {
            th.emplace_back(f, t);
        } catch (...) {
            break;
        }
    }
    for (int t = started; t < nt; t++) f(t);
    f(0);
    for (auto &x : th) x.join();
}

// Items of one run of oriented shell quartets, as the sequential planner
// would make them but with partial-sum offsets from 0.
struct PlanPart {
    std::vector<ShellGroup> groups;
    std::vector<ShellItem> tmp[kNB];
    std::vector<float> tcost[kNB];
    double units[kNB] = {}, flops[kNB] = {};
    int64_t npart = 0;
};

struct Orient {
    int su, sl;
    double cost;
};

void plan_items(const zv_context *c, const Orient *ors, size_t n, double budget, PlanPart &pp)
{
    const ClassInfo *ct = class_table();
    for (size_t q = 0; q < n; q++) {
        const Orient &o = ors[q];
        const int LU = c->h_sp_L[o.su], LL = c->h_sp_L[o.sl];
        const int ncu = c->h_sp_coff[o.su + 1] - c->h_sp_coff[o.su];
        const int ncl = c->h_sp_coff[o.sl + 1] - c->h_sp_coff[o.sl];
        const int npu = c->h_sp_np[o.su], npl = c->h_sp_np[o.sl];
        const int nk = nchunk(npl), nst = nstep(npu), nc = ncu * ncl;
        // slices of chunks first (they repeat the transform only), then of steps;
        // none shorter than 10 times the transform that it repeats: shorter ones
        // fill the chip no better and pay for it in partial sums (7 AOs 1.28 ms
        // at 3 times, 1.14 at 6, 1.05 at 10, 1.13 at 16; 45 AOs 22.5, 20.8, 20.4,
        // 19.8)
        const double least = 10.0 * transform_cost(LU, LL, ncu, ncl);
        const double want = std::ceil(o.cost / std::max(budget, least));
        const int kc = (int)std::min<double>(nk, std::max(1.0, want));
        const int ks = (int)std::min<double>(nst, std::max(1.0, std::ceil(want / kc)));
        const int np = npass(LU, LL);
        pp.groups.push_back(ShellGroup{o.su, o.sl, kc * ks * np, 0, pp.npart});
        const double pq = (double)npu * npl;
        for (int p = 0; p < np; p++) {
            const int b = bucket_of(LU, LL, p);
            const double cost = quartet_cost(ct[b], npu, npl) / (kc * ks);
            // algorithmic flops: Boys and R once per primitive quartet, one
            // multiply-add per needed (sigma, row)
            if (p == 0) pp.units[b] += pq;
            pp.flops[b] += pq * ((p == 0 ? boys_r_flops(LU + LL) : 0.0) + 2.0 * ct[b].acc);
            for (int i = 0; i < kc; i++)
                for (int j = 0; j < ks; j++) {
                    pp.tmp[b].push_back(ShellItem{o.su, o.sl, (int)((int64_t)nst * j / ks),
                                                  (int)((int64_t)nst * (j + 1) / ks),
                                                  (int)((int64_t)nk * i / kc),
                                                  (int)((int64_t)nk * (i + 1) / kc), pp.npart});
                    pp.tcost[b].push_back((float)cost);
                    pp.npart += nc;
                }
        }
    }
}

// Orientation, splitting and ordering of a list of shell quartets (x, y),
// both shell pairs of order <= ZV_LMAX_T with kept primitive pairs.  The
// uniform side is the pair of lower order (fewer sigma, so fewer
// accumulators per row), of equal ones the cheaper by padded steps and
// chunks.  Long lists are planned on host threads over contiguous runs of
// quartets whose items are joined in order, so the plan is the same for any
// thread count.
void plan_shell(const zv_context *c, const std::vector<std::pair<int, int>> &sq, Plan &pl,
                std::vector<char> &hbuf)
{
    using clk = std::chrono::steady_clock;
    auto ms_since = [](clk::time_point t) {
        return std::chrono::duration<double, std::milli>(clk::now() - t).count();
    };
    auto tt = clk::now();
    const size_t nq = sq.size();
    const int nt = plan_threads(nq);
    const ClassInfo *ct = class_table();
    std::vector<Orient> ors(nq);
    run_threads(nt, [&](int t) {
        for (size_t q = nq * t / nt; q < nq * (t + 1) / nt; q++) {
            int x = sq[q].first, y = sq[q].second;
            if (c->h_sp_L[x] > c->h_sp_L[y]) std::swap(x, y);
            const int LU = c->h_sp_L[x], LL = c->h_sp_L[y];
            auto cost = [&](int u, int l) {
                double s = transform_cost(LU, LL, c->h_sp_coff[u + 1] - c->h_sp_coff[u],
                                          c->h_sp_coff[l + 1] - c->h_sp_coff[l]);
                for (int p = 0; p < npass(LU, LL); p++)
                    s += quartet_cost(ct[bucket_of(LU, LL, p)], c->h_sp_np[u], c->h_sp_np[l]);
                return s;
            };
            const double cxy = cost(x, y), cyx = LU == LL && x != y ? cost(y, x) : cxy;
            ors[q] = cxy <= cyx ? Orient{x, y, cxy} : Orient{y, x, cyx};
        }
    });
    double total = 0.0;
    for (const Orient &o : ors) total += o.cost;
    // items of at most 1/20000 of the total cost: larger quartets are split,
    // so the sorted queue ends on short items (110 AOs 162.7 ms, with 1/40000
    // 164.7; 128-AO hydrocarbon 409.5 and 410.7)
    const double nitems =
        c->tune[ZV_TUNE_ERI_ITEMS] > 0 ? (double)c->tune[ZV_TUNE_ERI_ITEMS] : 20000.0;
    const double budget = std::max(total / nitems, 20000.0);
    pl.host_ms[0] = ms_since(tt);
    tt = clk::now();
    std::vector<PlanPart> parts(nt);
    run_threads(nt, [&](int t) {
        const size_t q0 = nq * t / nt, q1 = nq * (t + 1) / nt;
        plan_items(c, ors.data() + q0, q1 - q0, budget, parts[t]);
    });
    pl.host_ms[1] = ms_since(tt);
    tt = clk::now();
    // join the runs in order: partial-sum offsets shifted by the runs before
    pl.npart = 0;
    size_t ng = 0, nb_items[kNB] = {};
    for (const PlanPart &pp : parts) {
        ng += pp.groups.size();
        for (int b = 0; b < kNB; b++) nb_items[b] += pp.tmp[b].size();
    }
    size_t at = 0;
    for (int b = 0; b < kNB; b++) {
        pl.lo[b] = (int)at;
        at += nb_items[b];
    }
    pl.lo[kNB] = (int)at;
    hbuf.resize(sizeof(ShellItem) * at + sizeof(ShellGroup) * ng);
    pl.items = (ShellItem *)hbuf.data();
    pl.nitems = at;
    pl.groups = (ShellGroup *)(hbuf.data() + sizeof(ShellItem) * at);
    pl.ngroups = ng;
    std::vector<int64_t> off(nt, 0);
    std::vector<size_t> goff(nt, 0);
    for (int t = 0, g0 = 0; t < nt; t++) {
        PlanPart &pp = parts[t];
        off[t] = pl.npart;
        goff[t] = (size_t)g0;
        g0 += (int)pp.groups.size();
        for (int b = 0; b < kNB; b++) {
            pl.units[b] += pp.units[b];
            pl.flops[b] += pp.flops[b];
        }
        pl.npart += pp.npart;
    }
    run_threads(nt, [&](int t) {
        ShellGroup *dst = pl.groups + goff[t];
        for (ShellGroup g : parts[t].groups) {
            g.part += off[t];
            *dst++ = g;
        }
    });
    pl.host_ms[2] = ms_since(tt);
    tt = clk::now();
    // each bucket in descending cost (quarter-octave bins, counting sort), so the
    // long items start first and the queue ends on short ones; buckets are
    // independent and spread over the threads
    constexpr int NBIN = 256;
    static_assert(NBIN <= 256, "bins are stored as bytes");
    run_threads(nt, [&](int t) {
        std::vector<uint8_t> bin;
        std::vector<const ShellItem *> src;
        std::vector<float> cst;
        for (int b = t; b < kNB; b += nt) {
            const size_t n = nb_items[b];
            if (!n) continue;
            src.clear();
            cst.clear();
            std::vector<int64_t> shift;
            for (int u = 0; u < nt; u++)
                for (size_t i = 0; i < parts[u].tmp[b].size(); i++) {
                    src.push_back(&parts[u].tmp[b][i]);
                    cst.push_back(parts[u].tcost[b][i]);
                    shift.push_back(off[u]);
                }
            bin.resize(n);
            int cnt[NBIN + 1] = {};
            for (size_t i = 0; i < n; i++) {
                const int e = (int)std::floor(4.0 * std::log2(std::max(cst[i], 1.0f)));
                bin[i] = (uint8_t)(NBIN - 1 - std::min(e, NBIN - 1)); // large cost -> small bin
                cnt[bin[i] + 1]++;
            }
            for (int k = 0; k < NBIN; k++) cnt[k + 1] += cnt[k];
            for (size_t i = 0; i < n; i++) {
                ShellItem it = *src[i];
                it.part += shift[i];
                pl.items[pl.lo[b] + cnt[bin[i]]++] = it;
            }
        }
    });
    pl.host_ms[3] = ms_since(tt);
}

} // namespace

// ====================================================================== host
// Device layout of the shell-pair tables in b_spmeta: roff[nsp], goff[nsp]
// (int64), comp[npair], coff[nsp + 1], np[nsp], component -> shell pair
// [npair] (int); b_spu: primitive rows; b_spe: the two expansion tables.
static SPD spd_of(zv_context *c)
{
    const int64_t *d_roff = (const int64_t *)c->b_spmeta.p;
    const int64_t *d_goff = d_roff + c->nsp;
    const int *d_comp = (const int *)(d_goff + c->nsp);
    const int *d_coff = d_comp + c->npair;
    const int *d_np = d_coff + c->nsp + 1;
    const double *g = (const double *)c->b_spe.p;
    return SPD{d_comp, d_coff, d_np, d_roff, d_goff, (const double *)c->b_spu.p, g,
               g + c->sp_g_total};
}

// the Boys tables, made once per process, on the context's device (once per
// context)
int zv_boys_table(zv_context *c, const double **tab)
{
    static const std::vector<double> t = boys_table_host();
    ZV_CHECK(zv_ensure(c, c->b_btab, sizeof(double) * t.size()));
    *tab = (const double *)c->b_btab.p;
    if (c->btab_ready) return ZV_OK;
    ZV_HIPCHECK(c, hipMemcpyAsync(c->b_btab.p, t.data(), sizeof(double) * t.size(),
                                  hipMemcpyHostToDevice, c->stream));
    c->btab_ready = true;
    return ZV_OK;
}

int zv_shell_ready(zv_context *c, const PP &pp)
{
    const int nsp = c->nsp, np = c->npair;
    size_t meta = sizeof(int64_t) * 2 * nsp + sizeof(int) * (2 * (size_t)np + 2 * nsp + 1) + 64;
    ZV_CHECK(zv_ensure(c, c->b_spmeta, meta));
    if (c->sp_ready) return ZV_OK;
    // Z positions of every class and pass, once per context
    if (!c->ztab_ready) {
        const ClassInfo *ct = class_table();
        std::vector<short> all;
        c->h_ztab_off.assign(kNB, 0);
        for (int b = 0; b < kNB; b++) {
            c->h_ztab_off[b] = (int64_t)all.size();
            all.insert(all.end(), ct[b].ztab.begin(), ct[b].ztab.end());
        }
        ZV_CHECK(zv_ensure(c, c->b_ztab, sizeof(short) * all.size()));
        ZV_HIPCHECK(c, hipMemcpy(c->b_ztab.p, all.data(), sizeof(short) * all.size(),
                                 hipMemcpyHostToDevice));
        c->ztab_ready = true;
    }
    std::vector<int64_t> off(2 * (size_t)nsp);
    int64_t *roff = off.data(), *goff = roff + nsp;
    std::vector<int> tab;
    tab.reserve(2 * (size_t)np + 2 * nsp + 1);
    tab.insert(tab.end(), c->h_sp_comp.begin(), c->h_sp_comp.end());
    tab.insert(tab.end(), c->h_sp_coff.begin(), c->h_sp_coff.end());
    c->h_sp_np.assign(nsp, 0);
    int64_t r_tot = 0, g_tot = 0;
    for (int s = 0; s < nsp; s++) {
        const int c0 = c->h_sp_coff[s], nc = c->h_sp_coff[s + 1] - c0, L = c->h_sp_L[s];
        const int n = c->h_cnt[c->h_sp_comp[c0]];
        c->h_sp_np[s] = n;
        tab.push_back(n);
        roff[s] = r_tot;
        goff[s] = g_tot;
        if (L > ZV_LMAX_T) continue;
        r_tot += (int64_t)nchunk(n) * kLaneC * kRow[L];
        g_tot += (int64_t)nc * kG.t[L].n;
    }
    for (int s = 0; s < nsp; s++)
        for (int q = c->h_sp_coff[s]; q < c->h_sp_coff[s + 1]; q++) tab.push_back(s);
    ZV_CHECK(zv_ensure(c, c->b_spu, sizeof(double) * std::max<int64_t>(r_tot, 1)));
    ZV_CHECK(zv_ensure(c, c->b_spe, sizeof(double) * std::max<int64_t>(2 * g_tot, 1)));
    c->sp_g_total = g_tot;
    char *m = (char *)c->b_spmeta.p;
    ZV_HIPCHECK(c, hipMemcpyAsync(m, off.data(), sizeof(int64_t) * off.size(),
                                  hipMemcpyHostToDevice, c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(m + sizeof(int64_t) * off.size(), tab.data(),
                                  sizeof(int) * tab.size(), hipMemcpyHostToDevice, c->stream));
    const SPD sd = spd_of(c);
    {
        PhaseTimer tm(c, PH_PRIM);
        hipLaunchKernelGGL(k_pair_rows, dim3(nsp), dim3(128), 0, c->stream, pp, sd,
                           (double *)c->b_spu.p);
        ZV_HIPCHECK(c, hipGetLastError());
        hipLaunchKernelGGL(k_expansion, dim3(np), dim3(64), 0, c->stream, pp, sd, sd.np + nsp,
                           c->d_pair_i, c->d_pair_k, c->d_center, c->d_npower, c->d_itype,
                           (double *)c->b_spe.p, (double *)c->b_spe.p + g_tot);
        ZV_HIPCHECK(c, hipGetLastError());
    }
    ZV_HIPCHECK(c, hipStreamSynchronize(c->stream));
    c->sp_ready = true;
    return ZV_OK;
}

// Plan and launch the shell kernels of one Schwarz phase over the shell
// quartets sq; the partial sums stay in bpart for zv_shell_scatter.
int zv_shell_run(zv_context *c, const PP &pp, const std::vector<std::pair<int, int>> &sq,
                 DevBuf &bitem, DevBuf &bgroup, DevBuf &bpart, std::vector<char> &hplan,
                 int64_t *ngroups)
{
    using clk = std::chrono::steady_clock;
    const auto t0 = clk::now();
    Plan pl;
    plan_shell(c, sq, pl, hplan);
    const auto t1 = clk::now();
    *ngroups = (int64_t)pl.ngroups;
    if (!pl.nitems) return ZV_OK;
    const size_t bi = sizeof(ShellItem) * pl.nitems;
    const size_t bg = sizeof(ShellGroup) * pl.ngroups;
    const auto t2 = clk::now();
    ZV_CHECK(zv_ensure(c, bitem, bi));
    ZV_CHECK(zv_ensure(c, bgroup, bg));
    ZV_CHECK(zv_ensure(c, bpart, sizeof(double) * pl.npart));
    ZV_HIPCHECK(c, hipMemcpyAsync(bitem.p, hplan.data(), bi, hipMemcpyHostToDevice, c->stream));
    ZV_HIPCHECK(c, hipMemcpyAsync(bgroup.p, hplan.data() + bi, bg, hipMemcpyHostToDevice,
                                  c->stream));
    if (c->verbose) {
        const auto t3 = clk::now();
        auto ms = [](clk::duration d) { return std::chrono::duration<double, std::milli>(d).count(); };
        fprintf(stderr, "[zvmc] shell plan: %zu quartets -> %zu items, %zu groups; plan %.1f ms "
                "(orientation %.1f, items %.1f, join %.1f, bucket sort %.1f), device alloc + "
                "copy %.1f ms\n", sq.size(), pl.nitems, pl.ngroups, ms(t1 - t0), pl.host_ms[0],
                pl.host_ms[1], pl.host_ms[2], pl.host_ms[3], ms(t3 - t2));
    }
    const SPD sd = spd_of(c);
    const ClassInfo *ct = class_table();
    const ShellItem *di = (const ShellItem *)bitem.p;
    // The buckets write disjoint partial sums, so they run side by side on
    // the context's stream and its side streams (a bucket's last items leave
    // CUs idle that the next bucket fills), joined back before the scatter.
    // Most counted flops first, each to the stream with the fewest so far (the
    // count of a later pass leaves out the Boys values and R rows that it
    // repeats, so the passes of (3, 4) and (4, 4) come late).
    // bucket b = 50 pass + 5 LU + LL: statistics slot 36 + b
    static_assert(36 + kNB <= ZV_NSTAT, "statistics slots");
    constexpr int NST = 1 + zv_context::NSIDE;
    hipStream_t sts[NST] = {c->stream};
    for (int k = 0; k < zv_context::NSIDE; k++) sts[1 + k] = c->side[k];
    int order[kNB], nb = 0;
    for (int b = 0; b < kNB; b++)
        if (pl.lo[b + 1] > pl.lo[b]) order[nb++] = b;
    std::sort(order, order + nb, [&](int x, int y) { return pl.flops[x] > pl.flops[y]; });
    double load[NST] = {};
    // ZV_TUNE_ERI_STREAMS limits the streams (1: buckets one after another); a
    // single bucket needs no fork
    const int nst = nb == 1 ? 1
                    : c->tune[ZV_TUNE_ERI_STREAMS] > 0
                        ? (int)std::min<int64_t>(c->tune[ZV_TUNE_ERI_STREAMS], NST)
                        : NST;
    // phase time: one span around the fork and join; the buckets' own spans
    // overlap and only go to their statistics slots
    PhaseTimer wall(c, PH_ERI);
    if (nst > 1) {
        ZV_HIPCHECK(c, hipEventRecord(c->ev_fork, c->stream));
        for (int k = 0; k < nst - 1; k++)
            ZV_HIPCHECK(c, hipStreamWaitEvent(c->side[k], c->ev_fork, 0));
    }
    for (int t = 0; t < nb; t++) {
        const int b = order[t];
        const int n = pl.lo[b + 1] - pl.lo[b];
        const int cls = 36 + b;
        c->cls_pq[cls] += pl.units[b];
        c->cls_flops[cls] += pl.flops[b];
        int s = 0;
        for (int q = 1; q < nst; q++)
            if (load[q] < load[s]) s = q;
        load[s] += pl.flops[b];
        PhaseTimer tm(c, PH_N, cls, sts[s]);
        if (!ct[b].launch) return zv_fail(c, ZV_ERR_STATE, "no shell kernel for bucket %d", b);
        ct[b].launch(LaunchArgs{sd, di + pl.lo[b], n, pp.btab,
                                (const short *)c->b_ztab.p + c->h_ztab_off[b],
                                (double *)bpart.p, sts[s]});
        ZV_HIPCHECK(c, hipGetLastError());
    }
    for (int k = 0; k < nst - 1; k++) {
        ZV_HIPCHECK(c, hipEventRecord(c->ev_join[k], c->side[k]));
        ZV_HIPCHECK(c, hipStreamWaitEvent(c->stream, c->ev_join[k], 0));
    }
    return ZV_OK;
}

int zv_shell_scatter(zv_context *c, const DevBuf &bgroup, const DevBuf &bpart, int64_t ngroups,
                     const double *pre, double *tri)
{
    constexpr int64_t most = kLaunchThreads / 256;
    for (int64_t g = 0; g < ngroups; g += most) {
        hipLaunchKernelGGL(k_shell_scatter, dim3((unsigned)std::min(ngroups - g, most)), dim3(256),
                           0, c->stream, (const ShellGroup *)bgroup.p + g, spd_of(c),
                           (const double *)bpart.p, pre, tri);
        ZV_HIPCHECK(c, hipGetLastError());
    }
    return ZV_OK;
}

int zv_zero(zv_context *c, double *x, int64_t n)
{
    if (n <= 0) return ZV_OK;
    hipLaunchKernelGGL(k_zero, dim3(nblk(n, 256)), dim3(256), 0, c->stream, x, n);
    ZV_HIPCHECK(c, hipGetLastError());
    return ZV_OK;
}
