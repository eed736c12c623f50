"""Cosine terms whose phase is beyond FP64's resolution: no reduction brings it to
[-pi, pi], the sin/cos table's range, so the term is held at phase 0.  The value
of such a term is a cosine of some angle (at most its amplitude), and the likelihood
and its gradient are the numbers that belong to it; a phase that is not a number
stays none."""
import numpy as np
import pytest

from astroemperor_amd import JitterBlock, OffsetBlock, ReddModel, RVData, SinusoidBlock, SmartSetter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [50, 300])
@pytest.mark.parametrize("P,ph", [(100.0, 1e17), (100.0, -4e18), (1e-14, 0.3), (-1e-15, 0.3), (100.0, 1e300)])
def test_far_phase_is_some_cosine(P, ph, n):
    rng = np.random.default_rng(n)
    data = RVData.from_arrays([2450000.0 + np.sort(rng.uniform(0, 3000.0, n))], [rng.normal(size=n)],
                              [rng.uniform(1.0, 2.0, n)])
    ob, jb, sb = OffsetBlock(1), JitterBlock(1), SinusoidBlock(1)
    ss = SmartSetter(data.as_table())
    for b in (ob, jb, sb):
        ss(b)
    m = ReddModel([ob, jb, sb], data)
    amp = 7.0
    x = np.array([0.5, 1.0, P, amp, ph])
    mu, e2 = m.my_model(x)
    assert np.all(np.abs(mu - 0.5) <= amp * (1 + 1e-12))
    r = m.data.Y - mu
    want = -0.5 * np.sum(r * r / e2 + np.log(e2)) - 0.5 * n * np.log(2 * np.pi)
    for p in ("fp64", "mixed"):
        for which in ("single_pass", "two_pass"):
            m.set_grad_kernel(which)
            lnl, g = m.lnl_grad_batch(x[None], p)
            assert lnl[0] == pytest.approx(want, rel=1e-12)
            assert g[0, 0] == pytest.approx(np.sum(r / e2), rel=1e-9, abs=1e-9)
            assert g[0, 3] == pytest.approx(np.sum(r / e2 * (mu - 0.5)) / amp, rel=1e-9, abs=1e-9)
        assert m.lnl_batch(x[None], p)[0] == pytest.approx(want, rel=1e-12)
    x[4] = np.nan
    assert m.lnl_batch(x[None])[0] == -np.inf and m.lnl_grad_batch(x[None])[0][0] == -np.inf
