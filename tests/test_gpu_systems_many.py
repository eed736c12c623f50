"""A survey whose launches would hold 2^32 threads or more (from 2^18 systems on at
1024 walkers each) goes out in pieces: every system's first state is evaluated, and
after a sweep the last systems' walkers have moved and their stored likelihoods are
those of their positions."""
import numpy as np
import pytest

from astroemperor_amd import OffsetBlock, ReddModel, RVData, SmartSetter, SystemsPT

pytestmark = pytest.mark.gpu


def test_survey_beyond_2_32_threads():
    rng = np.random.default_rng(3)
    data = RVData.from_arrays([2450000.0 + np.array([0.0, 5.0, 9.0])], [np.array([-3.0, 1.0, 2.0])], [np.full(3, 2.0)])
    ob = OffsetBlock(1)
    SmartSetter(data.as_table())(ob)
    m = ReddModel([ob], data)
    kept = m.descriptor()
    m.descriptor = lambda: kept                       # one descriptor for all systems
    S, T, W = (1 << 18) + 3, 2, 512
    p0 = rng.normal(0.0, 1.0, size=(T, W, 1))

    def stored(x):                                    # a walker outside the prior has none
        x = x.reshape(-1, 1)
        return np.where(m.lnprior_batch(x) > -np.inf, m.lnl_batch(x), -np.inf).reshape(T, W)

    ref = stored(p0)
    y = SystemsPT([m] * S, T, W, [p0] * S, betas=np.array([1.0, 0.3]), seed=9, adapt_mode=-1)
    for s in (0, 1, S // 2, (1 << 17) - 1, 1 << 17, S - 4, S - 1):
        x, lnl, _ = y.state(s)
        assert np.array_equal(x, p0) and np.allclose(lnl, ref, rtol=1e-12, atol=0), s
    y.run(1, use_graph=False)
    y.run(1)
    acc = y.accepted.reshape(S, -1).sum(1)
    assert acc.min() > 0
    for s in (0, 1, S // 2, (1 << 17) - 1, 1 << 17, S - 4, S - 1):
        x, lnl, _ = y.state(s)
        assert not np.array_equal(x, p0), s
        assert np.allclose(lnl, stored(x), rtol=1e-12, atol=0), s
    y.close()
