"""Pair counts that one histogram could not hold in 32 bits.

A wave takes its histogram's counts to the 64-bit sums after 2^23 wave-iterations.
Two waves count every pair of 60,000 positions and 56,000 shapes in one bin
(3.36e9), private and deterministic; four waves
share a histogram of 480 bins.  Counts equal those of a full launch exactly, sums
within the rounding of as many additions.
"""
import numpy as np
import pytest

from measure_ia_amd import binning
from measure_ia_amd.engine import SampleArrays

pytestmark = pytest.mark.gpu

L = 20.0
N_POS, N_SHAPE = 60000, 56000


@pytest.fixture(scope="module")
def engine():
    from measure_ia_amd.engine import get_engine
    return get_engine(0)


@pytest.fixture(scope="module")
def sample():
    rng = np.random.default_rng(17)
    theta = rng.uniform(0.0, np.pi, N_SHAPE)
    return SampleArrays(positions=rng.uniform(0.0, L, (N_POS, 3)), shapes=rng.uniform(0.0, L, (N_SHAPE, 3)),
                        axis=np.stack([np.cos(theta), np.sin(theta)], 1), e=rng.uniform(0.0, 0.6, N_SHAPE),
                        boxsize=L, los=2)


@pytest.mark.parametrize("nr,n2,waves,det", [(1, 1, 2, 0), (1, 1, 2, 1), (12, 40, 4, 0)])
def test_spilled_counts(engine, sample, nr, n2, waves, det):
    print(nr, n2, waves, det, flush=True)
    r_bins = np.linspace(1e-9, 15.0, nr + 1)  # all separations: at most sqrt(200)
    th = binning.rppi_thresholds(r_bins, np.linspace(-10.0, 10.0, n2 + 1), 1e-9, 15.0)
    full = engine.count(sample, th, method="fast")
    few = engine.count(sample, th, method="fast", tuning={"waves": waves, "deterministic": det})
    assert few.stats["wave_iterations"] // waves > 1 << 23, few.stats  # every wave spills
    np.testing.assert_array_equal(few.npairs, full.npairs)
    np.testing.assert_array_equal(few.dd, full.npairs.astype(float))
    assert N_POS * N_SHAPE - 10 <= int(full.npairs[0].sum()) <= N_POS * N_SHAPE  # (pi = +10 exactly, r < 1e-9)
    # n additions round by at most n 2^-53 of the sum of the terms' sizes (e < 1: at most n)
    n = full.npairs[0].astype(float)
    assert np.all(np.abs(few.splus[0] - full.splus[0]) <= 1e-9 * n)
    assert np.all(np.abs(few.scross - full.scross) <= 1e-9 * n)
