"""Lightcone counts over numbers of patches, weights and shapes against the oracle.

Items are sorted by patch pair with counters in LDS up to 64 patches and by a
radix sort beyond, ranges are grouped by patch per block, and the histogram
slots differ for weighted and unweighted samples with and without shapes.
Counts and patch tallies equal the oracle's, sums within 1e-6.
"""
import numpy as np
import pytest

from measure_ia_amd import binning, synth
from oracle import lightcone as olc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_patches", [0, 1, 64, 65, 90])
@pytest.mark.parametrize("weights,shapes", [(True, True), (False, True), (True, False), (False, False)])
def test_patches_match_oracle(n_patches, weights, shapes):
    from measure_ia_amd.engine import LightconeArrays, get_engine
    from measure_ia_amd.lightcone import rotated_ellipticity
    print(n_patches, weights, shapes, flush=True)
    a = synth.lightcone(1200, 500, seed=n_patches + 7, weights=True, ra=(10.0, 20.0), dec=(-4.0, 4.0),
                        chi=(300.0, 700.0))
    patch = patch_s = None
    if n_patches:
        def of(ra, dec):
            return ((np.floor((ra - 10.0) * 9.7).astype(int) * 7 + np.floor((dec + 4.0) * 5.3).astype(int))
                    % n_patches).astype(np.int32)
        patch, patch_s = of(a["RA"], a["DEC"]), of(a["RA_shape_sample"], a["DEC_shape_sample"])
    w, ws = (a["weight"], a["weight_shape_sample"]) if weights else (None, None)
    c2, s2 = rotated_ellipticity(a["e1"], a["e2"]) if shapes else (None, None)
    rb, pb = np.logspace(np.log10(0.5), np.log10(15.0), 9), np.linspace(-20.0, 20.0, 11)
    lc = LightconeArrays(ra=a["RA"], dec=a["DEC"], chi=a["chi"], cos_dec=np.cos(a["DEC"] / 180 * np.pi),
                         ra_s=a["RA_shape_sample"], dec_s=a["DEC_shape_sample"], chi_s=a["chi_shape_sample"],
                         weight=w, weight_shape=ws, c2=c2, s2=s2, patch=patch, patch_s=patch_s, n_patches=n_patches)
    got = get_engine(0).count_lightcone(lc, binning.rppi_thresholds(rb, pb, 0.5, 15.0))
    kw = dict(e1=a["e1"], e2=a["e2"]) if shapes else {}
    if n_patches:
        kw.update(patch=patch, patch_s=patch_s, n_patches=n_patches)
    one, one_s = np.ones(len(a["RA"])), np.ones(len(a["RA_shape_sample"]))
    ref = olc.count("rppi", a["RA"], a["DEC"], a["chi"], w if weights else one, a["RA_shape_sample"],
                    a["DEC_shape_sample"], a["chi_shape_sample"], ws if weights else one_s, rb, pb, 0.5, 15.0, **kw)
    np.testing.assert_array_equal(got.npairs, np.asarray(ref["NP"]).reshape(got.npairs.shape))
    np.testing.assert_allclose(got.dd, np.asarray(ref["DD"]).reshape(got.dd.shape), rtol=1e-9, atol=1e-12)
    if not weights:
        np.testing.assert_array_equal(got.dd, got.npairs.astype(float))
    if shapes:
        ab = np.asarray(ref["SplusD_abs"]).reshape(got.splus.shape)
        err = np.abs(got.splus - np.asarray(ref["SplusD"]).reshape(got.splus.shape)) / (ab + 1e-300)
        assert err.max() <= 1e-6, err.max()
