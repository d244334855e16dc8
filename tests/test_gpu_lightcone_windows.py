"""Lightcone planning beyond the stencil cells whose windows are kept.

Up to 2^24 stencil cells the count pass keeps the shape windows for the emit pass;
beyond, the emit pass finds them again.  16,000 positions near the observer against
100,000 shapes over the sky have more (every block reaches every cell), each eighth of
the near ones has fewer, and the eighths' counts add up.
"""
import numpy as np
import pytest

from measure_ia_amd import binning

pytestmark = pytest.mark.gpu


def test_windows_found_again():
    from measure_ia_amd.engine import LightconeArrays, get_engine
    engine = get_engine(0)
    rng = np.random.default_rng(9)

    def sky(n):
        return rng.uniform(0.0, 360.0, n), np.degrees(np.arcsin(rng.uniform(-0.95, 0.95, n)))
    n, m, P = 16000, 100000, 27
    ra, dec = sky(n)
    far, far_dec = sky(20000)
    ra, dec = np.concatenate([ra, far]), np.concatenate([dec, far_dec])
    chi = np.concatenate([rng.uniform(4.0, 8.0, n), rng.uniform(2400.0, 2600.0, 20000)])
    ra_s, dec_s = sky(m)
    chi_s = rng.uniform(5.0, 25.0, m)

    def of(r, d):
        return ((r // 15.0).astype(int) * 5 + ((d + 90.0) // 36.0).astype(int)).astype(np.int32) % P
    patch, patch_s = of(ra, dec), of(ra_s, dec_s)
    th = binning.rppi_thresholds(np.logspace(np.log10(0.5), np.log10(20.0), 9), np.linspace(-20.0, 20.0, 11), 0.5,
                                 20.0)

    def count(sel):
        lc = LightconeArrays(ra=ra[sel], dec=dec[sel], chi=chi[sel], cos_dec=np.cos(dec[sel] / 180 * np.pi),
                             ra_s=ra_s, dec_s=dec_s, chi_s=chi_s, patch=patch[sel], patch_s=patch_s, n_patches=P)
        return engine.count_lightcone(lc, th)
    every = np.arange(len(ra))
    whole = count(every)
    parts = [count(every[(every >= n) | (every % 8 == k)]) for k in range(8)]
    far_only = count(every[every >= n])
    np.testing.assert_array_equal(whole.npairs + 7 * far_only.npairs, sum(p.npairs for p in parts))
    np.testing.assert_array_equal(whole.dd, whole.npairs.astype(float))
