"""The deterministic reduction where one key holds many slots.

Without regions every wave's histogram flush is a slot of one key.  Its slots are
summed in pieces of 32, so numbers of waves around the edges of pieces are
compared with the oracle and run twice for equal bits, and the finalisation of a
count without regions may not take many times that of one with regions.
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
@pytest.mark.parametrize("name", ["uniform_auto_nojk", "weighted_los0"])
def test_pieces_match_oracle(engine, name, mode):
    data, L, cfg = make_case(name)
    cfg = dict(cfg, L_sub=0)
    pr, ref, _ = oracle_counts(data, L, cfg, mode)
    p, sample = engine_sample(data, L, cfg)
    th = thresholds(cfg, L, mode)
    for waves in (1, 2, 31, 32, 33, 63, 64, 65, 129, 700, 0):
        print(name, mode, waves, flush=True)
        tu = {"deterministic": 1, "waves": waves}
        first = engine.count(sample, th, method="fast", variance=True, tuning=tu)
        compare(first, ref, p.R, 0, cfg["weights"])
        again = engine.count(sample, th, method="fast", variance=True, tuning=tu)
        for f in ("npairs", "dd", "splus", "scross", "variance"):
            np.testing.assert_array_equal(getattr(first, f), getattr(again, f))


def test_finalisation_without_regions(engine):
    rng = np.random.default_rng(3)
    data, L, cfg = make_case("uniform_jk27")
    data["Position"] = rng.uniform(0.0, L, (60000, 3))
    ms = {}
    for n in (0, 3):
        cfg = dict(cfg, L_sub=n, nr=10, n2=20)
        _, sample = engine_sample(data, L, cfg)
        th = thresholds(cfg, L, "rppi")
        ms[n] = min(engine.count(sample, th, tuning={"deterministic": 1}).stats["ms_finalize"] for _ in range(5))
    assert ms[0] < 8.0 * ms[3], ms
