"""The grid that the tuner picks where it once went wrong.

With pi_max of half the box, blocks as tall as the box make every pair take the
minimum image by itself; with few shapes in a large volume, small cells leave
blocks of three shapes.  The counts on the picked grids equal those on others.
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


def _sample(n_pos, n_shape, L, seed):
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0.0, L, (n_pos, 3))
    theta = rng.uniform(0.0, np.pi, n_shape)
    return SampleArrays(positions=pos, shapes=pos[:n_shape].copy(),
                        axis=np.stack([np.cos(theta), np.sin(theta)], 1), e=rng.uniform(0.0, 0.6, n_shape),
                        boxsize=L, los=2)


def _count(engine, s, r_max, n_r, pi_max, tuning=None):
    r_bins, pi_bins, _ = prep.bin_edges(0.1, r_max, n_r, 20, pi_max, s.boxsize)
    return engine.count(s, binning.rppi_thresholds(r_bins, pi_bins, 0.1, r_max), tuning=tuning)


def test_blocks_are_low_where_the_reach_is_half_the_box(engine):
    s = _sample(100001, 50003, 75.0, 1)
    got = _count(engine, s, 20.0, 10, 37.5)
    tall = _count(engine, s, 20.0, 10, 37.5, {"columns_per_side": 30, "slabs_per_side": 4, "slabs_per_block": 4})
    assert 4 * got.stats["slabs_per_block"] <= got.stats["slabs_per_side"], got.stats
    np.testing.assert_array_equal(got.npairs, tall.npairs)


def test_blocks_hold_several_shapes_in_thin_samples(engine):
    s = _sample(562663, 40378, 300.0, 2)
    got = _count(engine, s, 30.0, 8, 60.0)
    other = _count(engine, s, 30.0, 8, 60.0, {"columns_per_side": 14, "slabs_per_side": 8, "slabs_per_block": 2})
    st = got.stats
    cells = st["columns_per_side"] ** 2 * (st["slabs_per_side"] // st["slabs_per_block"])
    assert 40378 / cells > 4.5, st
    np.testing.assert_array_equal(got.npairs, other.npairs)
