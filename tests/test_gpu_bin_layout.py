"""Histogram bins of every sum layout against the FP64 oracle.

A bin holds two sums (S+D, SxD), a third for weights (DD) or variances (sum of
e+^2), or both.  With three sums the pair counts lie in front of the sums, padded
to 8 bytes for odd numbers of bins, otherwise inside the bin.  Odd and even
numbers of bins, a single bin, and enough bins for several passes over r are
counted with private (deterministic) and shared histograms in both modes.
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
@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("variance", [False, True])
@pytest.mark.parametrize("nr,n2", [(1, 1), (3, 5), (4, 6), (12, 30), (9, 101)])
def test_layouts_match_oracle(engine, nr, n2, variance, weights, mode):
    data, L, cfg = make_case("uniform_jk27")
    cfg = dict(cfg, nr=nr, n2=n2, weights=weights)
    if weights:
        rng = np.random.default_rng(nr * 1000 + n2)
        data["weight"] = rng.uniform(0.5, 1.5, len(data["Position"]))
        data["weight_shape_sample"] = rng.uniform(0.5, 1.5, len(data["Position_shape_sample"]))
    pr, ref, _ = oracle_counts(data, L, cfg, mode)
    p, sample = engine_sample(data, L, cfg)
    th = thresholds(cfg, L, mode)
    for tu in (None, {"waves": 5}, {"deterministic": 1}):
        print(nr, n2, variance, weights, mode, tu, flush=True)
        res = engine.count(sample, th, method="fast", variance=variance, tuning=tu)
        compare(res, ref, p.R, 27, weights)
        if variance:
            v = res.variance / (2 * p.R) ** 2
            assert np.all(np.abs(v - ref["variance"]) <= 1e-6 * np.maximum(ref["variance"], 1e-300))
