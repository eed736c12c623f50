"""Models without planets, whose likelihood is bound by its loads (pairs of epochs at
once, times only where a term needs them, fewer waves per vector), and columns at
odd positions (systems packed one after another), against the oracle: series
around one and two lanes' pairs and chunks, with and without an acceleration, a
sinusoid and a moving average, at the rule's and at every number of waves."""
import numpy as np
import pytest

from astroemperor_amd import (AccelerationBlock, JitterBlock, KeplerianBlock, MOAVBlock, OffsetBlock, ReddModel, RVData,
                              SinusoidBlock, SmartSetter, SystemsPT)
from tests.conftest import oracle_for

pytestmark = pytest.mark.gpu


def _star(n, k=0, acc=0, sin=0, ma=None):
    rng = np.random.default_rng(n)
    counts = [n - n // 3, n // 3] if n > 5 else [n]
    bjd = [np.sort(2450000.0 + rng.uniform(0.0, 500.0, c)) for c in counts]
    data = RVData.from_arrays(bjd, [rng.normal(0.0, 5.0, c) + np.arange(c) % 2 for c in counts],
                              [rng.uniform(1.0, 3.0, c) for c in counts])
    I = len(counts)
    blocks = [KeplerianBlock(1, p + 1) for p in range(k)] + ([AccelerationBlock(acc)] if acc else [])
    blocks += [OffsetBlock(I), JitterBlock(I)]
    blocks += [MOAVBlock(I, {"order": 1, "global": ma == "global"})] if ma else []
    blocks += [SinusoidBlock(1)] if sin else []
    ss = SmartSetter(data.as_table())
    for b in blocks:
        ss(b)
    return ReddModel(blocks, data, semantics="intended")


def _draws(m, n, rng):
    lim = m.limits_free()
    th = lim[:, 0] + (lim[:, 1] - lim[:, 0]) * rng.uniform(0.3, 0.7, size=(n, len(lim)))
    for j, nm in enumerate(m.names_free()):
        if nm.startswith("Acceleration"):
            th[:, j] *= 1e-2
    return th


@pytest.mark.parametrize("terms", [dict(), dict(acc=1), dict(sin=1), dict(ma="instrument"), dict(ma="global", acc=2)])
@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 127, 128, 129, 257, 1025])
def test_batched_likelihood(n, terms):
    m = _star(n, **terms)
    o = oracle_for(m)
    th = _draws(m, 6, np.random.default_rng(n + 1))
    ref = np.array([o.my_likelihood(x) for x in th])
    for w in (0, 1, 2, 4, 8):
        m.set_waves_per_theta(w)
        for p in ("fp64", "mixed"):
            assert np.allclose(m.lnl_batch(th, p), ref, rtol=1e-10, atol=0), (w, p)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_systems_at_odd_positions(precision):
    rng = np.random.default_rng(4)
    models = [_star(n, k=k) for n, k in [(3, 0), (64, 1), (65, 0), (67, 1), (129, 2), (131, 0), (7, 1), (256, 1)]]
    p0 = [_draws(m, 2 * 8, rng).reshape(2, 8, -1) for m in models]
    y = SystemsPT(models, 2, 8, p0, precision=precision, seed=1)
    for s, (m, x) in enumerate(zip(models, p0)):
        o = oracle_for(m)
        _, lnl, lnp = y.state(s)
        for t in range(2):
            for w in range(8):
                want = o.my_likelihood(x[t, w]) if lnp[t, w] > -np.inf else -np.inf
                assert lnl[t, w] == pytest.approx(want, rel=1e-10, abs=0.0 if precision == "fp64" else 1e-6), (s, t, w)
