"""Counts whose launch keeps a histogram per wave, against the plain kernel.

Counts of fewer than 1.6e9 expected candidate pairs share a histogram per workgroup.
Here 60,000 positions and 40,000 shapes reach most of a box of 30 (2.3e9), so every
wave has its own and claims tail chunks: both modes, with and without weights
and variances, against the brute-force kernel, pair counts equal and sums within
the rounding of their additions.
"""
import numpy as np
import pytest

from measure_ia_amd import binning
from measure_ia_amd.engine import SampleArrays
from oracle import prep

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from measure_ia_amd.engine import get_engine
    return get_engine(0)


def _sample(weights, los):
    rng = np.random.default_rng(23)
    n, m, L = 60000, 40000, 30.0
    pos, shp = rng.uniform(0.0, L, (n, 3)), rng.uniform(0.0, L, (m, 3))
    theta = rng.uniform(0.0, np.pi, m)
    w, ws = (rng.uniform(0.5, 1.5, n), rng.uniform(0.5, 1.5, m)) if weights else (None, None)
    return SampleArrays(positions=pos, shapes=shp, axis=np.stack([np.cos(theta), np.sin(theta)], 1),
                        e=rng.uniform(0.0, 0.6, m), weight=w, weight_shape=ws, boxsize=L, los=los, jk_per_side=2,
                        jk_sub=L / 2)


@pytest.mark.parametrize("mode", ["rppi", "rmu"])
@pytest.mark.parametrize("weights", [False, True])
def test_private_histograms_match_plain(engine, weights, mode):
    print(mode, weights, flush=True)
    s = _sample(weights, 1 if mode == "rmu" and weights else 2)
    r_max = 14.0 if mode == "rppi" else 16.0
    r_bins, pi_bins, mu_bins = prep.bin_edges(0.1, r_max, 10, 16, 15.0, 30.0)
    th = (binning.rppi_thresholds(r_bins, pi_bins, 0.1, r_max) if mode == "rppi"
          else binning.rmu_thresholds(r_bins, mu_bins, 0.1, r_max))
    ref = engine.count(s, th, method="plain", variance=True)
    assert ref.npairs[0].sum() > 9e8
    for tu, variance in ((None, True), (None, False), ({"waves": 48}, True), ({"waves": 4096}, False)):
        got = engine.count(s, th, method="fast", variance=variance, tuning=tu)
        np.testing.assert_array_equal(got.npairs, ref.npairs)
        # n additions of terms below 2.25 (weights) round by at most n 2^-53 of the sum of their sizes
        n = 2.25 * ref.npairs.astype(float)
        assert np.all(np.abs(got.dd - ref.dd) <= 1e-9 * n)
        assert np.all(np.abs(got.splus - ref.splus) <= 1e-9 * n)
        assert np.all(np.abs(got.scross - ref.scross) <= 1e-9 * n[0])
        if variance:
            assert np.all(np.abs(got.variance - ref.variance) <= 1e-9 * 2.25 * n[0])
