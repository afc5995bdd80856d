"""The shell-quartet ERI kernels against the CPU oracle at the edges of their
tiles: the number of kept primitive pairs of a shell pair (ng^2 for AOs on one
centre) below, at and above the step of 4 uniform-side and the chunk of 16
lane-side primitive pairs, for every pair of shell-pair orders 0..4, each
reached by products of different shells (p x p, d x s and r^2-type s x s are
all of order 2)."""
import numpy as np
import pytest

from slater_stoch_amd import basis as B

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from slater_stoch_amd.zvmc import Engine
    e = Engine(0)
    yield e
    e.close()


# 1, 4, 9, 16, 25 and 49 primitive pairs on one centre; the tolerance is that
# of the other comparisons with the oracle (its polynomial recursion loses
# digits relative to the largest integral, not to each one)
@pytest.mark.parametrize("ng", [1, 2, 3, 4, 5, 7])
def test_shell_kernels_at_tile_edges(engine, oracle, ng):
    geom = B.geometry_from_angstrom(["O", "H"], [[0.05, -0.1, 0.2], [0.7, 0.4, -0.5]])
    basis = {"O": [("1S", 2.6), ("2S", 1.9), ("2P", 2.1), ("3D", 1.7)],
             "H": [("1S", 1.2), ("3P", 1.4), ("4F", 1.8)]}
    bas = B.expand_basis(geom, basis, ng0=ng)
    engine.set_basis(bas)
    eri, pre, _ = engine.gauss_eri()
    orders = {key[1:3] for key in engine.eri_stats() if key[0] == "shell"}
    assert orders == {(a, b) for a in range(5) for b in range(a, 5)}
    q = B.quartet_mapping(bas.n)
    rng = np.random.default_rng(ng)
    keep = np.flatnonzero(np.abs(pre[q[2] - 1, q[0] - 1] * pre[q[3] - 1, q[1] - 1]) >= 1e-30)
    pick = rng.choice(keep, 2500, replace=False)
    oracle.set_basis(bas)
    ref, _ = oracle.gauss_eri([a[pick] for a in q], None)
    np.testing.assert_allclose(eri[pick], ref, rtol=1e-10, atol=1e-12 * np.abs(ref).max())


# lists short enough for the largest split of a quartet over waves (more waves
# than the one or 16 primitive pairs of a pair), of mixed splits and with
# classes of one wave per quartet; f x f pairs reach the runtime-order kernel
@pytest.mark.parametrize("nq,ng", [(1, 4), (40, 1), (40, 4), (1500, 7), (60000, 2)])
def test_list_classes_side_by_side(engine, nq, ng):
    geom = B.geometry_from_angstrom(["O", "H"], [[0.05, -0.1, 0.2], [0.7, 0.4, -0.5]])
    basis = {"O": [("1S", 2.6), ("2S", 1.9), ("2P", 2.1), ("3D", 1.7)],
             "H": [("1S", 1.2), ("3P", 1.4), ("4F", 1.8)]}
    bas = B.expand_basis(geom, basis, ng0=ng)
    engine.set_basis(bas)
    eri, _, _ = engine.gauss_eri()
    qi, qj, qk, ql = B.quartet_mapping(bas.n)
    full = np.empty((bas.n + 1,) * 4)
    for a, b in ((qi, qk), (qk, qi)):
        for c, d in ((qj, ql), (ql, qj)):
            full[a, b, c, d] = eri
            full[c, d, a, b] = eri
    rng = np.random.default_rng(nq)
    i, k, j, l = rng.integers(1, bas.n + 1, (4, nq))
    got = engine.gauss_ijkl(i, k, j, l)
    # the tolerance of the other comparison of the two sets of kernels
    np.testing.assert_allclose(got, full[i, k, j, l], rtol=1e-12,
                               atol=1e-15 * np.abs(eri).max())
    np.testing.assert_array_equal(engine.gauss_ijkl(i, k, j, l), got)
    if nq <= 16384:
        np.testing.assert_array_equal(engine.gauss_ijkl_noalloc(i, k, j, l), got)


def test_hermite_planes_on_first_use(engine):
    """The component kernels' Hermite coefficients are made on first use: by
    the allocation-free entry point after gauss_eri, by a list, and again for
    a new basis, with the same values."""
    geom = B.geometry_from_angstrom(["O", "H"], [[0.05, -0.1, 0.2], [0.7, 0.4, -0.5]])
    basis = {"O": [("2S", 1.9), ("2P", 2.1), ("3P", 1.3)], "H": [("1S", 1.2), ("3D", 1.4)]}
    bas = B.expand_basis(geom, basis, ng0=3)
    rng = np.random.default_rng(3)
    q = rng.integers(1, bas.n + 1, (4, 300))
    engine.set_basis(bas)
    engine.gauss_eri()
    first = engine.gauss_ijkl_noalloc(*q)
    engine.set_basis(B.expand_basis(geom, basis, ng0=2))
    other = engine.gauss_ijkl(*q)
    engine.set_basis(bas)
    np.testing.assert_array_equal(engine.gauss_ijkl(*q), first)
    assert np.abs(other - first).max() > 1e-6
