"""bench.py's share of matrix instructions in the analytic phase's counted
flops: rows that need one scaled Hermite weight are plain vector multiply-adds,
and the multiply-adds it splits are those that the library counts."""
import math

import numpy as np
import pytest

import bench
from slater_stoch_amd import configs


def boys_r_flops(l):
    """Boys values, R table and prefactor per primitive quartet of order l."""
    return 25 + 3 * (l + 1) + 4 * (math.comb(l + 4, 4) - 1) + 12


# vector share of the row sums: rows of the top order need one weight.  (1, 1):
# rows of orders 0, 1 need 3 weights, the six of order 2 one, 6 / 18; (0, L):
# one weight everywhere; pass 3 of (4, 4): the rows of order 8 need one
@pytest.mark.parametrize("lu,ll,p,share", [(0, 3, 0, 1.0), (1, 1, 0, 6 / 18), (1, 2, 0, 10 / 40),
                                           (1, 3, 0, 15 / 75), (4, 4, 3, 1.0)])
def test_vector_rows_are_not_matrix_work(lu, ll, p, share):
    boys_r = boys_r_flops(lu + ll)
    stats = {("shell", lu, ll, p + 1, False): dict(units=10.0, flops=10.0 * (boys_r + 100.0))}
    want = (1.0 - share) * 100.0 / (boys_r + 100.0)
    assert bench.mfma_fraction(dict(eri_stats=stats)) == pytest.approx(want, rel=1e-12, abs=0.0)


@pytest.mark.gpu
def test_multiply_adds_are_the_librarys():
    from slater_stoch_amd.zvmc import Engine
    bas = configs.random_molecule(seed=3, n_heavy=2, n_h=1)
    with Engine(0) as eng:
        eng.set_basis(bas)
        eng.gauss_eri(device_only=True)
        st = {k: v for k, v in eng.eri_stats().items() if k[0] == "shell"}
    assert {k[1:3] for k in st} == {(a, b) for b in range(5) for a in range(b + 1)}
    for (_, lu, ll, p, _), v in st.items():
        pq = st["shell", lu, ll, 1, False]["units"]
        boys_r = boys_r_flops(lu + ll) if p == 1 else 0.0
        assert v["units"] == (pq if p == 1 else 0.0)
        macs = sum(bench.quartet_macs(lu, ll, p - 1))
        np.testing.assert_allclose(v["flops"], pq * (boys_r + 2.0 * macs), rtol=1e-12)
