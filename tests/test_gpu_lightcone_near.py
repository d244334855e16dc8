"""Lightcone counts with positions near the observer and many patches.

At a few Mpc a block of positions reaches the whole sky and holds hundreds to tens
of thousands of shape ranges, which are grouped by patch through counters in LDS
beyond 256.  Counts, tallies and sums against the oracle, in both modes and with
patch numbers on either side of the items' radix sort; and the planning time of
60,000 near shapes, which must not grow with the square of a block's ranges.
"""
import numpy as np
import pytest

from measure_ia_amd import binning
from measure_ia_amd.synth import ellipticity_noise
from oracle import lightcone as olc

pytestmark = pytest.mark.gpu


def _sky(rng, n):
    return rng.uniform(0.0, 360.0, n), np.degrees(np.arcsin(rng.uniform(-0.95, 0.95, n)))


def _sample(n_near, n_far, m, n_patches, seed=1):
    from measure_ia_amd.engine import LightconeArrays
    from measure_ia_amd.lightcone import rotated_ellipticity
    rng = np.random.default_rng(seed)
    n = n_near + n_far
    ra, dec = _sky(rng, n)
    chi = np.concatenate([rng.uniform(4.0, 8.0, n_near), rng.uniform(2400.0, 2600.0, n_far)])
    ra_s, dec_s = _sky(rng, m)
    chi_s = rng.uniform(5.0, 25.0, m)
    e12 = ellipticity_noise(rng, m, 0.25)
    c2, s2 = rotated_ellipticity(e12[:, 0], e12[:, 1])

    def of(r, d):
        return ((r // 15.0).astype(int) * 5 + ((d + 90.0) // 36.0).astype(int)).astype(np.int32) % n_patches
    patches = {} if n_patches == 0 else dict(patch=of(ra, dec), patch_s=of(ra_s, dec_s), n_patches=n_patches)
    lc = LightconeArrays(ra=ra, dec=dec, chi=chi, cos_dec=np.cos(dec / 180 * np.pi), ra_s=ra_s, dec_s=dec_s,
                         chi_s=chi_s, weight=rng.uniform(0.5, 1.5, n), weight_shape=rng.uniform(0.5, 1.5, m),
                         c2=c2, s2=s2, **patches)
    return lc, e12


RB = np.logspace(np.log10(0.5), np.log10(20.0), 9)


def _bins(mode):
    if mode == "rppi":
        second = np.linspace(-20.0, 20.0, 11)
        return second, binning.rppi_thresholds(RB, second, 0.5, 20.0)
    second = np.linspace(-1.0, 1.0, 11)
    return second, binning.rmu_thresholds(RB, second, 0.5, 20.0)


@pytest.mark.parametrize("mode", ["rppi", "rmu"])
@pytest.mark.parametrize("n_patches", [1, 27, 70])
def test_near_blocks_match_oracle(n_patches, mode):
    from measure_ia_amd.engine import get_engine
    print(n_patches, mode, flush=True)
    lc, e12 = _sample(70, 1500, 6000, n_patches)
    second, th = _bins(mode)
    got = get_engine(0).count_lightcone(lc, th)
    ref = olc.count(mode, lc.ra, lc.dec, lc.chi, lc.weight, lc.ra_s, lc.dec_s, lc.chi_s, lc.weight_shape, RB, second,
                    0.5, 20.0, e1=e12[:, 0], e2=e12[:, 1], patch=lc.patch, patch_s=lc.patch_s, n_patches=n_patches)
    np.testing.assert_array_equal(got.npairs, np.asarray(ref["NP"]).reshape(got.npairs.shape))
    np.testing.assert_allclose(got.dd, np.asarray(ref["DD"]).reshape(got.dd.shape), rtol=1e-9, atol=1e-12)
    for have, name in ((got.splus, "SplusD"), (got.scross, "ScrossD")):
        ab = np.asarray(ref[name + "_abs"]).reshape(-1, *have.shape[-2:])[: len(have) if have.ndim == 3 else 1]
        want = np.asarray(ref[name]).reshape(-1, *have.shape[-2:])[: len(have) if have.ndim == 3 else 1]
        err = np.abs(have.reshape(want.shape) - want) / (ab + 1e-300)
        assert err.max() <= 1e-6, (name, err.max())


def test_planning_time_of_near_blocks():
    from measure_ia_amd.engine import get_engine
    engine = get_engine(0)
    _, th = _bins("rppi")
    lc, _ = _sample(64, 20000, 60000, 27)
    ms = min(engine.count_lightcone(lc, th).stats["ms_plan"] for _ in range(5))
    assert ms < 10.0, ms
