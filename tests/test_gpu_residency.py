"""The pair kernel launches no more workgroups than a CU's LDS holds at once.

LDS is allocated in granules of 1,280 bytes.  A histogram of 45 x 49 bins with the
edges of 90 x 49 makes workgroups of 54,096 bytes, of which two fit (55,040 bytes
each); a third one would run behind them.
"""
import numpy as np
import pytest
import torch

from paircases import engine_sample, make_case, thresholds

pytestmark = pytest.mark.gpu


def test_waves_fit_the_lds():
    from measure_ia_amd.engine import get_engine
    engine = get_engine(0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    data, L, cfg = make_case("uniform_jk27")
    cfg = dict(cfg, nr=90, n2=49)
    _, sample = engine_sample(data, L, cfg)
    th = thresholds(cfg, L, "rppi")
    counts = []
    for rows, per_cu in ((45, 2), (44, 3), (20, 6)):
        res = engine.count(sample, th, method="fast", tuning={"r_bins_per_pass": rows})
        print(rows, res.stats["waves"], flush=True)
        assert res.stats["waves"] <= per_cu * 4 * cus, res.stats
        counts.append(res.npairs)
    for c in counts[1:]:
        np.testing.assert_array_equal(c, counts[0])
