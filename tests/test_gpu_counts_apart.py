"""Histograms of two and four sums with the pair counts in front of the sums.

A row of weighted r bins with variances that fits LDS only with 36 bytes a bin, not
with the usual 40, is counted by the batched kernel, alone and in a batch, and
deterministic counts take the narrower bins where they save passes.  Every output is compared with
the FP64 oracle.
"""
import numpy as np
import pytest

from paircases import compare, engine_sample, make_case, oracle_counts, thresholds

pytestmark = pytest.mark.gpu


def run(mode, weights, nr, n2, deterministic):
    from measure_ia_amd.engine import get_engine
    engine = get_engine(0)
    data, L, cfg = make_case("uniform_jk27")
    cfg = dict(cfg, nr=nr, n2=n2, weights=weights)
    if weights:
        rng = np.random.default_rng(n2)
        data["weight"] = rng.uniform(0.5, 1.5, len(data["Position"]))
        data["weight_shape_sample"] = rng.uniform(0.5, 1.5, len(data["Position_shape_sample"]))
    _, ref, _ = oracle_counts(data, L, cfg, mode)
    p, sample = engine_sample(data, L, cfg)
    th = thresholds(cfg, L, mode)
    tuning = {"deterministic": deterministic}
    for variance in {weights, False}:
        print(mode, weights, variance, nr, n2, deterministic, flush=True)
        single = engine.count(sample, th, method="fast", variance=variance, tuning=tuning)
        assert single.stats["method"] == 1  # not the plain kernel
        for res in [single] + engine.count_batch([sample, sample], th, variance=variance, tuning=tuning):
            compare(res, ref, p.R, 27, weights)
            if variance:
                v = res.variance / (2 * p.R) ** 2
                assert np.all(np.abs(v - ref["variance"]) <= 1e-6 * np.maximum(ref["variance"], 1e-300))


@pytest.mark.parametrize("mode", ["rppi", "rmu"])
@pytest.mark.parametrize("weights,nr,n2", [(False, 60, 60), (False, 33, 101), (True, 33, 101), (True, 101, 33), (False, 256, 256)])
def test_deterministic_passes(mode, weights, nr, n2):
    run(mode, weights, nr, n2, 1)


def test_narrow_bins_save_passes():
    """100 x 20 bins: one pass of four waves per CU (four of 24-byte bins do not fit)."""
    from measure_ia_amd.engine import get_engine
    engine = get_engine(0)
    data, L, cfg = make_case("uniform_jk27")
    _, sample = engine_sample(data, L, cfg)
    th = thresholds(dict(cfg, nr=100, n2=20), L, "rppi")
    one = engine.count(sample, th, method="fast", tuning={"deterministic": 1, "r_bins_per_pass": 100})
    own = engine.count(sample, th, method="fast", tuning={"deterministic": 1})
    assert own.stats["wave_iterations"] == one.stats["wave_iterations"]
    np.testing.assert_array_equal(own.npairs, one.npairs)
