"""Monte Carlo blocks run in rounds: the means and standard errors of a call
that takes several blocks per round, one, or several chunks per block equal
those formed from the block means of a block-by-block run on the same
samples."""
import numpy as np
import pytest

from slater_stoch_amd import configs
from slater_stoch_amd.zvmc import TUNE_EST_SPLIT, TUNE_MC_CHUNK

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from slater_stoch_amd.zvmc import Engine
    e = Engine(0)
    yield e
    e.close()


# chunk 0: automatic (all blocks in one round); 160: several chunks per block
# of 200 or 360 samples; 400: rounds of 10 and of 2 blocks with a rest; split
# 7 leaves uneven and, for the shortest block, empty splits
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nbl,npts,chunk,split", [(1, 40, 0, 0), (10, 40, 0, 0), (7, 40, 0, 7),
                                                  (3, 200, 160, 0), (5, 360, 160, 7),
                                                  (5, 200, 400, 0), (12, 40, 400, 2),
                                                  (3, 1000, 0, 64)])
def test_rounds_equal_block_by_block(engine, precision, nbl, npts, chunk, split):
    engine.set_basis(configs.water_minimal(ng0=6))
    _, _, blk = engine.mc_blocks(nbl, npts, precision, seed=5, stream=2, block_means=True)
    try:
        engine.set_tuning(TUNE_MC_CHUNK, chunk)
        engine.set_tuning(TUNE_EST_SPLIT, split)
        mean, err = engine.mc_blocks(nbl, npts, precision, seed=5, stream=2)
    finally:
        engine.set_tuning(TUNE_MC_CHUNK, 0)
        engine.set_tuning(TUNE_EST_SPLIT, 0)
    # the FP32 stage sums of 8 samples are the same in every form; sums of at
    # most 1000 FP64 terms in another order differ by less than 1e-13 of the
    # largest block mean's scale
    scale = np.abs(blk).max()
    want = blk.mean(0)
    np.testing.assert_allclose(mean, want, rtol=1e-12, atol=1e-13 * scale)
    var = np.abs((blk ** 2).mean(0) - want ** 2)
    np.testing.assert_allclose(err ** 2 * nbl, var, rtol=1e-9, atol=1e-13 * scale ** 2)
