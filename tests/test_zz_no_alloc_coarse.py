"""mia_count_noalloc where the tuner's grid needs more than the static workspace.

A million positions and shapes in a box of 75 fit only on a coarser grid; the counts
equal mia_count's.
"""
import ctypes

import numpy as np
import pytest

from measure_ia_amd import _capi, binning
from measure_ia_amd.engine import SampleArrays

pytestmark = pytest.mark.gpu


def test_noalloc_takes_a_coarser_grid():
    from measure_ia_amd.engine import get_engine
    eng = get_engine(0)
    rng = np.random.default_rng(2)
    L, n = 75.0, 1_000_000
    pos = rng.uniform(0.0, L, (n, 3))
    theta = rng.uniform(0.0, np.pi, n)
    s = SampleArrays(positions=pos, shapes=pos, axis=np.stack([np.cos(theta), np.sin(theta)], 1),
                     e=rng.uniform(0.0, 0.6, n), boxsize=L, los=2, jk_per_side=3, jk_sub=L / 3)
    th = binning.rppi_thresholds(np.logspace(-1.0, np.log10(20.0), 11), np.linspace(-37.5, 37.5, 21), 0.1, 20.0)
    ms, keep, _ = eng._prepare(s)
    bins, keep_b = eng._bins(th, False)
    layout, buf, c = eng._outputs(27, th.n_r * th.n_2, False)
    stream = eng.torch.cuda.current_stream(eng.dev).cuda_stream
    rc = eng.lib.mia_count_noalloc(eng.ctx, ctypes.byref(ms), ctypes.byref(bins), ctypes.byref(c), None,
                                   ctypes.c_void_p(stream))
    _capi.check(eng.lib, eng.ctx, rc)
    got = eng._host((layout, buf), 27, th, {})
    ref = eng.count(s, th, method="fast")
    np.testing.assert_array_equal(got.npairs, ref.npairs)
    assert np.abs(got.splus - ref.splus).max() <= 1e-12 * np.abs(ref.splus).max()
