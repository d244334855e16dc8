"""Lightcone S+D and SxD in both modes on either side of the items' radix sort.

Items are sorted by patch pair with counters in LDS up to 64 patches and by a radix
sort beyond; S+D and SxD, their tallies, counts and DD against the oracle.
"""
import numpy as np
import pytest

from measure_ia_amd import binning, synth
from oracle import lightcone as olc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["rppi", "rmu"])
@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("n_patches", [64, 65])
def test_sums_match_oracle(n_patches, weights, mode):
    from measure_ia_amd.engine import LightconeArrays, get_engine
    from measure_ia_amd.lightcone import rotated_ellipticity
    print(n_patches, weights, mode, flush=True)
    a = synth.lightcone(1500, 600, seed=n_patches, weights=True, ra=(10.0, 20.0), dec=(-4.0, 4.0), chi=(300.0, 700.0))

    def of(ra, dec):
        return ((np.floor((ra - 10.0) * 9.7).astype(int) * 7 + np.floor((dec + 4.0) * 5.3).astype(int))
                % n_patches).astype(np.int32)
    patch, patch_s = of(a["RA"], a["DEC"]), of(a["RA_shape_sample"], a["DEC_shape_sample"])
    w, ws = (a["weight"], a["weight_shape_sample"]) if weights else (None, None)
    c2, s2 = rotated_ellipticity(a["e1"], a["e2"])
    rb = np.logspace(np.log10(0.5), np.log10(15.0), 9)
    second = np.linspace(-20.0, 20.0, 11) if mode == "rppi" else np.linspace(-1.0, 1.0, 11)
    th = (binning.rppi_thresholds if mode == "rppi" else binning.rmu_thresholds)(rb, second, 0.5, 15.0)
    lc = LightconeArrays(ra=a["RA"], dec=a["DEC"], chi=a["chi"], cos_dec=np.cos(a["DEC"] / 180 * np.pi),
                         ra_s=a["RA_shape_sample"], dec_s=a["DEC_shape_sample"], chi_s=a["chi_shape_sample"],
                         weight=w, weight_shape=ws, c2=c2, s2=s2, patch=patch, patch_s=patch_s, n_patches=n_patches)
    got = get_engine(0).count_lightcone(lc, th)
    one, one_s = np.ones(len(a["RA"])), np.ones(len(a["RA_shape_sample"]))
    ref = olc.count(mode, a["RA"], a["DEC"], a["chi"], w if weights else one, a["RA_shape_sample"],
                    a["DEC_shape_sample"], a["chi_shape_sample"], ws if weights else one_s, rb, second, 0.5, 15.0,
                    e1=a["e1"], e2=a["e2"], patch=patch, patch_s=patch_s, n_patches=n_patches)
    np.testing.assert_array_equal(got.npairs, np.asarray(ref["NP"]).reshape(got.npairs.shape))
    np.testing.assert_allclose(got.dd, np.asarray(ref["DD"]).reshape(got.dd.shape), rtol=1e-9, atol=1e-12)
    for have, name in ((got.splus, "SplusD"), (got.scross, "ScrossD")):
        want = np.asarray(ref[name]).reshape(-1, *have.shape[-2:])
        ab = np.asarray(ref[name + "_abs"]).reshape(want.shape)
        have = have.reshape(-1, *have.shape[-2:])
        err = np.abs(have - want[: len(have)]) / (ab[: len(have)] + 1e-300)
        assert err.max() <= 1e-6, (name, err.max())
