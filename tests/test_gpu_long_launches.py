"""Work lists longer than one launch holds (2^32 threads; a longer launch runs
only the remainder): one class of a quartet list with a wavefront per quartet,
and a molecule of so many shells that the shell kernels have a wavefront and
the sums of their slices a workgroup for each of more than 2^32 / 64 shell
quartets."""
import numpy as np
import pytest

from slater_stoch_amd import basis as B
from slater_stoch_amd import configs

pytestmark = pytest.mark.gpu

ONE_LAUNCH = 2 ** 32 // 64  # wavefronts


@pytest.fixture(scope="module")
def engine():
    from slater_stoch_amd.zvmc import Engine
    e = Engine(0)
    yield e
    e.close()


def test_one_class_of_a_quartet_list(engine):
    bas = configs.water_minimal(ng0=2)
    engine.set_basis(bas)
    s = np.flatnonzero((bas.npower.sum(1) == 0) & (bas.i_type == 1)) + 1  # order 0
    rng = np.random.default_rng(4)
    head = rng.choice(s, (50, 4))
    row = rng.integers(0, 50, ONE_LAUNCH + 1000, dtype=np.int8)
    want = engine.gauss_ijkl(*head.T)
    got = engine.gauss_ijkl(*[head[:, x].astype(np.int32)[row] for x in range(4)])
    # the short list splits its quartets: 16 terms in another order
    np.testing.assert_allclose(got, want[row], rtol=1e-12, atol=1e-15 * np.abs(want).max())


def test_shell_quartets_of_many_shells(engine):
    # 153 s shells: 11,781 shell pairs, 69,401,871 shell quartets
    rng = np.random.default_rng(9)
    grid = np.stack(np.meshgrid(*[np.arange(6.0)] * 3), -1).reshape(-1, 3)[:153]
    geom = B.geometry_from_angstrom(["H"] * 153, 0.25 * grid + rng.uniform(-0.05, 0.05, (153, 3)))
    bas = B.expand_basis(geom, {"H": [("1S", 1.2)]}, ng0=1)
    assert bas.nint > ONE_LAUNCH
    engine.set_basis(bas)
    eri, pre, _ = engine.gauss_eri()
    i, j, k, l = B.quartet_mapping(bas.n)
    pick = rng.choice(i.size, 20000, replace=False)
    i, j, k, l = i[pick], j[pick], k[pick], l[pick]
    assert np.abs(pre).min() ** 2 >= 1e-30  # every quartet passes the Schwarz test
    ref = engine.gauss_ijkl(i, k, j, l)
    np.testing.assert_allclose(eri[pick], ref, rtol=1e-12, atol=1e-15 * np.abs(ref).max())
