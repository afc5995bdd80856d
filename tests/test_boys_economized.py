"""The economized Boys expansions of boys_table (csrc/eri_device.h), restated
here and checked on the CPU against the Boys function summed in extended
precision, at random T, at the ends of the expansions' intervals and at the
change to the complete integral.  Tolerance: the scheme's truncation (6e-18) and
about two roundings per order of the recursion, 8 x 1.1e-16 x 2 = 1.8e-15."""
import numpy as np
import pytest

LD = np.longdouble
M = 20
TMAX = [36.0, 40.0, 43.5, 46.5, 49.5, 52.0, 36.0, 36.0, 36.0]

FACT = np.cumprod([LD(1)] + [LD(k) for k in range(1, M + 1)])
CHEB = [[1], [0, 1]]
for _k in range(2, M + 1):
    _a = [0] + [2 * x for x in CHEB[-1]]
    for _t, _x in enumerate(CHEB[-2]):
        _a[_t] -= _x
    CHEB.append(_a)


def boys_exact(m_max, T):
    T = LD(T)
    s = term = LD(1) / (2 * m_max + 1)
    j = 0
    while term >= LD(1e-22) * s:
        j += 1
        term = term * 2 * T / (2 * m_max + 2 * j + 1)
        s += term
    e = np.exp(-T)
    F = [LD(0)] * m_max + [s * e]
    for m in range(m_max - 1, -1, -1):
        F[m] = (2 * T * F[m + 1] + e) / (2 * m + 1)
    return F


def expansion(L, T0, delta, deg):
    F = boys_exact(L + M, T0)
    q = [(-1) ** k * F[L + k] / FACT[k] * LD(delta) ** k for k in range(M + 1)]
    for k in range(M, deg, -1):
        a = q[k] / CHEB[k][k]
        for j, x in enumerate(CHEB[k]):
            q[j] -= a * x
    q = [q[k] / LD(delta) ** k for k in range(deg + 1)]
    if not 1 <= L <= 5:
        return [float(x) for x in q]
    return [float(F[L - 1])] + [float(-x / (k + 1)) for k, x in enumerate(q)]


def scheme(L, T):
    inv_h, deg = (4, 8) if L <= 4 else (2, 10)
    pair = 1 <= L <= 5
    F = [0.0] * (L + 1)
    if T < TMAX[L]:
        i = int(T * inv_h + 0.5)
        d = T - i / inv_h
        c = expansion(L, i / inv_h, 0.5 / inv_h, deg)
        b0, b1 = c[-1], 0.0
        for k in range(len(c) - 2, -1, -1):
            b1 = b0 if k == len(c) - 2 else b1 * d + b0
            b0 = b0 * d + c[k]
        if L == 0:
            return [b0]
        if pair:
            F[L - 1], F[L] = b0, -b1
            e = 2.0 * T * b1 + (2 * L - 1) * b0
        else:
            F[L], e = b0, np.exp(-T)
            F[L - 1] = (2.0 * T * F[L] + e) * (1.0 / (2 * L - 1))
        for m in range(L - 2, -1, -1):
            F[m] = (2.0 * T * F[m + 1] + e) * (1.0 / (2 * m + 1))
        return F
    F[0] = 0.5 / np.sqrt(T) * np.sqrt(np.pi)
    e = 0.0 if pair or T > 80.0 else np.exp(-T)
    for m in range(L):
        F[m + 1] = (F[m] * (2 * m + 1) - e) * (0.5 / T)
    return F


@pytest.mark.parametrize("L", range(9))
def test_economized_expansions(L):
    rng = np.random.default_rng(L)
    h = 0.25 if L <= 4 else 0.5
    edges = (np.array([0.0, 1.0, 7.0, 35.0]) + 0.5) * h
    t = TMAX[L]
    Ts = np.concatenate([rng.uniform(0.0, t, 60), rng.uniform(t, t + 60.0, 20), [0.0], edges,
                         np.nextafter(edges, 0.0), [np.nextafter(t, 0.0), t, 80.0, 81.0]])
    for T in Ts:
        ref = boys_exact(L, T)
        for m, f in enumerate(scheme(L, float(T))):
            assert abs(float(LD(f) / ref[m] - 1)) < 1.8e-15, (T, m)
