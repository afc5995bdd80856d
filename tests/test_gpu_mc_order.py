"""Progress lines and block means leave the Monte Carlo results alone: mean and
standard error are the same bits with and without either, and they are the
statistics of the block means that are returned.  The basis has s, p and d
shells (units of one, three and six components) in few tiles, so that blocks
are split over the samples; the chunk of 400 makes rounds of several blocks
and a rest, that of 160 several chunks per block."""
import numpy as np
import pytest

from slater_stoch_amd import configs
from slater_stoch_amd.zvmc import TUNE_MC_CHUNK

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from slater_stoch_amd.zvmc import Engine
    e = Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("mode", ["philox", "fixed"])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16"])
@pytest.mark.parametrize("nbl,npts,chunk", [(10, 1000, 0), (7, 40, 0), (11, 120, 400),
                                            (3, 200, 160)])
def test_same_bits_with_progress_lines_and_block_means(engine, precision, mode, nbl, npts, chunk,
                                                       capfd):
    engine.set_basis(configs.random_molecule(seed=3, n_heavy=1, n_h=2))
    samples = engine.draw_samples(nbl * npts, seed=5, stream=2) if mode == "fixed" else None

    def run(verbose=0, **kw):
        engine._check(engine.lib.zv_set_verbose(engine.h, verbose))
        return engine.mc_blocks(nbl, npts, precision, samples=samples, seed=5, stream=2, **kw)

    try:
        engine.set_tuning(TUNE_MC_CHUNK, chunk)
        mean, err = run()
        mean_b, err_b, blk = run(block_means=True)
        capfd.readouterr()
        mean_v, err_v = run(2)
        lines = [x for x in capfd.readouterr().out.splitlines() if "MC block" in x]
        mean_vb, err_vb, blk_v = run(2, block_means=True)
    finally:
        engine.set_tuning(TUNE_MC_CHUNK, 0)
        engine._check(engine.lib.zv_set_verbose(engine.h, 0))
    assert np.any(mean != 0.0)
    for m, e in ((mean_b, err_b), (mean_v, err_v), (mean_vb, err_vb)):
        np.testing.assert_array_equal(m, mean)
        np.testing.assert_array_equal(e, err)
    np.testing.assert_array_equal(blk_v, blk)
    assert [int(x.split()[2]) for x in lines] == list(range(1, nbl + 1))
    # the statistics of the block means, added in block order
    s1, s2 = np.zeros(mean.size), np.zeros(mean.size)
    for x in blk:
        s1 += x
        s2 += x * x
    np.testing.assert_array_equal(mean, s1 / nbl)
    np.testing.assert_allclose(err, np.sqrt(np.abs(s2 / nbl - (s1 / nbl) ** 2)) / np.sqrt(nbl),
                               rtol=1e-14)


# each block of a round against a call of its own on the same samples: the first
# of several blocks starts at 0, the others bstride samples further each
@pytest.mark.parametrize("mode", ["philox", "fixed"])
@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16"])
@pytest.mark.parametrize("nbl,npts,chunk", [(7, 1000, 0), (10, 40, 0), (11, 120, 400)])
def test_blocks_of_a_round_equal_calls_of_their_own(engine, precision, mode, nbl, npts, chunk):
    engine.set_basis(configs.random_molecule(seed=3, n_heavy=1, n_h=2))
    samples = engine.draw_samples(nbl * npts, seed=5, stream=2)
    try:
        engine.set_tuning(TUNE_MC_CHUNK, chunk)
        _, _, blk = engine.mc_blocks(nbl, npts, precision, seed=5, stream=2, block_means=True,
                                     samples=samples if mode == "fixed" else None)
    finally:
        engine.set_tuning(TUNE_MC_CHUNK, 0)
    # the FP32 stage sums of 8 samples are the same in both; at most 1000 FP64
    # terms in another order differ by less than 1e-13 of the largest block mean
    scale = np.abs(blk).max()
    for b in range(nbl):
        part = [a[b * npts:(b + 1) * npts] for a in samples]
        alone, _ = engine.mc_blocks(1, npts, precision, samples=part)
        np.testing.assert_allclose(blk[b], alone, rtol=1e-12, atol=1e-13 * scale)
