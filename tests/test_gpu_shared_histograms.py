"""Shared histograms and thin position columns against the FP64 oracle.

600 (r_p, pi) or (r, mu) bins leave LDS for so few private histograms that the
waves of a workgroup share one, taking the items of a key from a counter.  The
counts are compared with oracle.brute (pair counts and tallies equal, sums
within 1e-6) with full workgroups, with 1, 3 and 6 waves (workgroups with idle
waves, and many keys per group), and with one position column per item (columns
without positions, and the tails of positions on jackknife faces).
"""
import numpy as np
import pytest

from paircases import compare, engine_sample, make_case, oracle_counts, thresholds

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from measure_ia_amd.engine import get_engine
    return get_engine(0)


@pytest.mark.parametrize("mode", ["rppi", "rmu"])
@pytest.mark.parametrize("name", ["uniform_jk27", "clustered_jk8", "open_box_jk27", "lattice_boundaries"])
def test_shared_histograms_match_oracle(engine, name, mode):
    data, L, cfg = make_case(name)
    cfg = dict(cfg, nr=15, n2=40)
    pr, ref, _ = oracle_counts(data, L, cfg, mode)
    p, sample = engine_sample(data, L, cfg)
    th = thresholds(cfg, L, mode)
    K = cfg["L_sub"] ** 3 if cfg["L_sub"] else 0
    base = engine.count(sample, th, method="fast")
    compare(base, ref, p.R, K, cfg["weights"])
    for tu in ({"waves": 1}, {"waves": 3}, {"waves": 6}, {"item_positions": 1},
               {"item_positions": 1, "waves": 6}, {"deterministic": 1}):
        print(name, mode, tu, flush=True)
        res = engine.count(sample, th, method="fast", tuning=tu)
        np.testing.assert_array_equal(res.npairs, base.npairs)
        compare(res, ref, p.R, K, cfg["weights"])
