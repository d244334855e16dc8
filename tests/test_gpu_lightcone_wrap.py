"""Lightcone statistics and counts beyond 2^32 in one workgroup or wave.

Four waves of one workgroup bin 4.3e9 pairs on the exact path (a thin shell, whose
bin guesses are never accepted): the recheck statistic equals the number of pairs.
"""
import numpy as np
import pytest

from measure_ia_amd import binning

pytestmark = pytest.mark.gpu

N = 65600  # N^2 = 4303360000 > 2^32


def _count(ra, ra_s, r_bins, n_2, waves, **kw):
    from measure_ia_amd.engine import LightconeArrays, get_engine
    rng = np.random.default_rng(3)
    n, m = len(ra), len(ra_s)
    dec, dec_s = 1e-9 * rng.uniform(-1.0, 1.0, n), 1e-9 * rng.uniform(-1.0, 1.0, m)
    chi, chi_s = rng.uniform(1000.0, 1010.0, n), rng.uniform(1000.0, 1010.0, m)
    lc = LightconeArrays(ra=ra, dec=dec, chi=np.full(n, 1000.0) if kw.get("flat") else chi,
                         cos_dec=np.cos(dec / 180 * np.pi), ra_s=ra_s, dec_s=dec_s, chi_s=chi_s)
    th = binning.rppi_thresholds(r_bins, np.linspace(-20.0, 20.0, n_2 + 1), r_bins[0], r_bins[-1])
    return get_engine(0).count_lightcone(lc, th, tuning={"waves": waves})


def test_rechecks_beyond_32_bits():
    # all positions at one point, all shapes 10.005 Mpc away from them
    sep = np.degrees(10.005 / 1000.0)
    rng = np.random.default_rng(5)
    ra = 10.0 + 1e-9 * rng.uniform(-1.0, 1.0, N)
    ra_s = 10.0 + sep + 1e-9 * rng.uniform(-1.0, 1.0, N)
    res = _count(ra, ra_s, np.logspace(np.log10(10.0), np.log10(10.01), 11), 8, 4, flat=True)
    assert int(res.npairs[0].sum()) == N * N
    assert res.stats["rechecks"] == N * N, res.stats


def test_counts_beyond_32_bits():
    """One wave counts 4.3e9 pairs in one bin."""
    rng = np.random.default_rng(6)
    res = _count(10.0 + rng.uniform(0.0, 1.0, N), 10.0 + rng.uniform(0.0, 1.0, N), np.array([1e-12, 100.0]), 1, 1)
    assert int(res.npairs[0].sum()) == N * N
    np.testing.assert_array_equal(res.dd, res.npairs.astype(float))
