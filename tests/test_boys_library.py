"""The Boys table that the library builds and the evaluation that its kernels
run (csrc/boys_table.h, compiled here for the host) against the series in
extended precision, at random T, at the ends of the expansions' intervals and
at the change to the complete integral.

Tolerance, in units u = 1.1e-16 of one rounding: below boys_tmax the two Horner
results carry 1.5 u, the difference that replaces exp(-T) 2.5 u more, and each
order downward, a mean of two positive terms, 1.5 u: with 8 orders at most
16 u = 1.8e-15.  Above it F_0 carries 2.5 u and each order upward 4 u (its
factor: the square of the reciprocal root 2.5 u, two products)."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "slater_stoch_amd" / "csrc"
U = 2.0 ** -53
LD = np.longdouble

DRIVER = r"""
#include <cstdio>
#include "boys_table.h"
using namespace zveri;
template <int L> void run(const std::vector<double> &t, int n, const double *T)
{
    for (int x = 0; x < n; x++) {
        double F[L + 1];
        boys_table<L>(T[x], t.data() + boys_off(L), F);
        for (int m = 0; m <= L; m++) printf("%d %d %a %a %d\n", L, m, T[x], F[m], T[x] < boys_tmax(L));
    }
}
int main()
{
    const std::vector<double> t = boys_table_host();
    if (t.size() != (size_t)boys_off(kBoysLmax + 1)) return 1;
    std::vector<double> T;
    for (double x; scanf("%la", &x) == 1;) T.push_back(x);
    const int n = (int)T.size();
    run<0>(t, n, T.data());
    run<1>(t, n, T.data());
    run<2>(t, n, T.data());
    run<3>(t, n, T.data());
    run<4>(t, n, T.data());
    run<5>(t, n, T.data());
    run<6>(t, n, T.data());
    run<7>(t, n, T.data());
    run<8>(t, n, T.data());
    return 0;
}
"""


def series(T, m_max=8):
    """F_0 .. F_m_max at T: the series of the highest order, then downward."""
    T = LD(T)
    s = term = LD(1) / (2 * m_max + 1)
    j = 0
    while term >= LD(1e-23) * s:
        j += 1
        term = term * 2 * T / (2 * m_max + 2 * j + 1)
        s += term
    e = np.exp(-T)
    F = [LD(0)] * m_max + [s * e]
    for m in range(m_max - 1, -1, -1):
        F[m] = (2 * T * F[m + 1] + e) / (2 * m + 1)
    return F


def test_library_table_against_the_series(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("no hipcc")
    (tmp_path / "driver.hip").write_text(DRIVER)
    exe = tmp_path / "driver"
    subprocess.run([hipcc, "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off",
                    f"-I{CSRC}", str(tmp_path / "driver.hip"), "-o", str(exe)], check=True)
    rng = np.random.default_rng(12)
    # every interval: its grid point, both ends and a point inside
    grid = np.arange(0.0, 52.25, 0.125)
    tmax = np.array([36.0, 40.0, 43.5, 46.5, 49.5, 52.0])
    T = np.concatenate([grid, np.nextafter(grid[1:], 0.0), rng.uniform(0.0, 52.0, 600), tmax,
                        np.nextafter(tmax, 0.0), rng.uniform(36.0, 120.0, 200),
                        [1e-300, 1e-20, 1e-8, 80.0, np.nextafter(80.0, 81.0), 1e3, 1e5]])
    out = subprocess.run([str(exe)], input="\n".join(float(t).hex() for t in T), text=True,
                         capture_output=True, check=True).stdout.splitlines()
    assert len(out) == 45 * T.size
    exact = {float(t): series(t) if t <= 200.0 else None for t in T}
    for line in out:
        L, m, t, f, inside = line.split()
        L, m, t, f = int(L), int(m), float.fromhex(t), float.fromhex(f)
        if exact[t] is None:  # the complete integral, Gamma(m + 1/2) / (2 T^(m + 1/2))
            ref = np.sqrt(LD("3.14159265358979323846264338327950288")) / (2 * np.sqrt(LD(t)))
            for k in range(m):
                ref = ref * (2 * k + 1) / (2 * LD(t))
        else:
            ref = exact[t][m]
        tol = 16 * U if inside == "1" else (2.5 + 4 * m) * U
        assert abs(float(LD(f) / ref - 1)) < tol, (L, m, t)
