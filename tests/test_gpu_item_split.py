"""Work items split over waves and workgroups against the FP64 oracle.

The pair kernel's shares begin and end inside items (at a batch of 64 of an
item's positions), and the waves of a workgroup with a shared histogram take an
item in quarters where the workgroup has few items.  Items as large as they get
are counted by few and by many waves, in private (deterministic) and shared
histograms, and the time of the pair kernel must not hang on the items' size.
"""
import numpy as np
import pytest

from measure_ia_amd import binning
from measure_ia_amd.engine import SampleArrays
from measure_ia_amd.synth import clustered, ellipticity_noise
from oracle import prep
from paircases import compare, engine_sample, make_case, oracle_counts, thresholds

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from measure_ia_amd.engine import get_engine
    return get_engine(0)


@pytest.mark.parametrize("mode", ["rppi", "rmu"])
@pytest.mark.parametrize("name", ["uniform_auto_nojk", "clustered_jk8", "reach_beyond_half_box",
                                  "lattice_boundaries"])
def test_split_items_match_oracle(engine, name, mode):
    data, L, cfg = make_case(name)
    pr, ref, _ = oracle_counts(data, L, cfg, mode)
    p, sample = engine_sample(data, L, cfg)
    K = cfg["L_sub"] ** 3 if cfg["L_sub"] else 0
    th = thresholds(cfg, L, mode)
    n = cfg["L_sub"] or 1
    big = {"item_positions": 1 << 20, "columns_per_side": 2 * n, "slabs_per_side": 2 * n}
    for tu in ({}, big, {"item_positions": 1 << 20}):
        for waves in (1, 2, 3, 7, 40, 700, 0):
            for det in (0, 1):
                t = dict(tu, waves=waves, deterministic=det)
                print(name, mode, t, flush=True)
                res = engine.count(sample, th, method="fast", tuning=t)
                compare(res, ref, p.R, K, cfg["weights"])


def test_pair_time_does_not_hang_on_item_size(engine):
    """20,000 clustered galaxies and 5,000 shapes in a box of 75: few, large items
    took three times as long as small ones while a wave worked on whole items."""
    L = 75.0
    cat = clustered(20000, 5000, L, 100, 1.0, 40, 0.2, 0.2, seed=5)
    pos, shp = cat.data["Position"], cat.data["Position_shape_sample"]
    rng = np.random.default_rng(5)
    e12 = ellipticity_noise(rng, len(shp), 0.25)
    theta = 0.5 * np.arctan2(e12[:, 1], e12[:, 0])
    sample = SampleArrays(positions=pos, shapes=shp, axis=np.stack([np.cos(theta), np.sin(theta)], 1),
                          e=np.linalg.norm(e12, axis=1), weight=rng.uniform(0.5, 1.5, len(pos)),
                          weight_shape=rng.uniform(0.5, 1.5, len(shp)), boxsize=L, los=2)
    r_bins, pi_bins, _ = prep.bin_edges(0.1, 20.0, 10, 20, 37.5, L)
    th = binning.rppi_thresholds(r_bins, pi_bins, 0.1, 20.0)
    best = {}
    for positions in (64, 1 << 20):
        for _ in range(10):
            ms = engine.count(sample, th, tuning={"item_positions": positions}).stats["ms_pairs"]
            best[positions] = min(ms, best.get(positions, ms))
    assert best[1 << 20] < 1.5 * best[64], best
