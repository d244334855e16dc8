"""Deterministic counts whose item order needs two sorts.

Sixteen samples with 4,096 regions each have 2^28 planner keys, and 203,000 shape
blocks each: key, block and rectangle exceed 64 bits and are sorted in two steps.
Counts equal those of the default path, and two runs give the same bits.
"""
import numpy as np
import pytest

from measure_ia_amd import binning
from measure_ia_amd.engine import SampleArrays

pytestmark = pytest.mark.gpu


def test_two_sorts():
    from measure_ia_amd.engine import get_engine
    engine = get_engine(0)
    rng = np.random.default_rng(8)
    L, n, m = 128.0, 300, 200000
    samples = []
    for _ in range(16):
        theta = rng.uniform(0.0, np.pi, m)
        samples.append(SampleArrays(positions=rng.uniform(0.0, L, (n, 3)), shapes=rng.uniform(0.0, L, (m, 3)),
                                    axis=np.stack([np.cos(theta), np.sin(theta)], 1), e=rng.uniform(0.0, 0.6, m),
                                    boxsize=L, los=2, jk_per_side=16, jk_sub=L / 16))
    th = binning.rppi_thresholds(np.array([0.5, 4.0]), np.array([-5.0, 5.0]), 0.5, 4.0)
    tu = {"columns_per_side": 128, "slabs_per_side": 128, "slabs_per_block": 1}
    ref = engine.count_batch(samples, th, tuning=tu)
    first = engine.count_batch(samples, th, tuning=dict(tu, deterministic=1))
    again = engine.count_batch(samples, th, tuning=dict(tu, deterministic=1))
    for a, b, c in zip(first, again, ref):
        assert a.npairs[0].sum() > 1000
        np.testing.assert_array_equal(a.npairs, c.npairs)
        assert np.all(np.abs(a.splus - c.splus) <= 1e-12 * (1.0 + c.npairs))
        for f in ("npairs", "dd", "splus", "scross", "region_stats"):
            np.testing.assert_array_equal(getattr(a, f), getattr(b, f))
