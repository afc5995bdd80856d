"""A quartet list of more than 2^32 / 64 = 67,108,864 quartets (a launch of more
than 2^32 threads runs only the remainder) in several classes, three of them so
short that their quartets are split over wavefronts."""
import numpy as np
import pytest

from slater_stoch_amd import configs

pytestmark = pytest.mark.gpu


def test_long_list_with_a_short_class():
    from slater_stoch_amd.zvmc import Engine
    bas = configs.water_minimal(ng0=2)
    order = bas.npower.sum(1)
    s, p = np.flatnonzero(order == 0) + 1, np.flatnonzero(order == 1) + 1
    n_ss, n_ps = 40_000_000, 27_200_000
    # (s s|s s), (p s|s s) and, in the middle, three quartets of other classes
    head = np.array([[s[0], s[1], s[2], s[0]], [p[0], s[0], s[1], s[2]], [p[0], p[0], p[1], p[1]],
                     [p[1], p[1], s[1], s[0]], [p[2], p[2], p[2], p[2]]], np.int32)
    counts = [n_ss, n_ps, 1, 1, 1]
    row = np.concatenate([np.full(n_ss, 0, np.int8), [2, 3, 4], np.full(n_ps, 1, np.int8)])
    assert sum(counts) > 2 ** 32 // 64 and max(counts) < 2 ** 32 // 64
    with Engine(0) as eng:
        eng.set_basis(bas)
        want = eng.gauss_ijkl(*head.T)
        got = eng.gauss_ijkl(*[head[:, x][row] for x in range(4)])
    # the short list splits every quartet: 16 or fewer terms in another order
    np.testing.assert_allclose(got, want[row], rtol=1e-12, atol=1e-15 * np.abs(want).max())
