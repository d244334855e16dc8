"""Passes over r bins of large binnings.

Every pass tests all candidate pairs again, so a pass of few waves per CU is better
than many passes of many.  The number of passes is the ratio of the pair kernel's
wave-iterations to those of a count in two passes; the counts are the same.
"""
import numpy as np
import pytest

from paircases import engine_sample, make_case, thresholds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("deterministic,most", [(1, 8), (0, 3)])
def test_few_passes(deterministic, most):
    from measure_ia_amd.engine import get_engine
    engine = get_engine(0)
    data, L, cfg = make_case("uniform_jk27")
    cfg = dict(cfg, nr=100, n2=100)
    _, sample = engine_sample(data, L, cfg)
    th = thresholds(cfg, L, "rppi")
    two = engine.count(sample, th, method="fast", tuning={"deterministic": deterministic, "r_bins_per_pass": 50})
    own = engine.count(sample, th, method="fast", tuning={"deterministic": deterministic})
    passes = 2.0 * own.stats["wave_iterations"] / two.stats["wave_iterations"]
    print(deterministic, passes, flush=True)
    assert passes <= most, passes
    np.testing.assert_array_equal(own.npairs, two.npairs)
