"""Batches whose launch would hold 2^32 threads or more (2^25 vectors at two waves
per vector, from 1024 epochs on) go out in pieces: the likelihood and both adjoints
of 2^25 + 3 vectors that repeat with a period of 1000 repeat with it, bit for bit,
and the first ones are those of a small batch."""
import numpy as np
import pytest
import torch

from astroemperor_amd import OffsetBlock, ReddModel, RVData, SmartSetter

pytestmark = pytest.mark.gpu


def test_likelihood_and_adjoints_beyond_2_32_threads():
    n, B, period = 1024, (1 << 25) + 3, 1000
    rng = np.random.default_rng(2)
    data = RVData.from_arrays([2450000.0 + np.sort(rng.uniform(0.0, 3000.0, n))], [rng.normal(size=n)], [np.full(n, 1.5)])
    ob = OffsetBlock(1)
    SmartSetter(data.as_table())(ob)
    m = ReddModel([ob], data)
    x = (torch.arange(B, device="cuda", dtype=torch.float64) % period * 1e-2)[:, None]
    few = m.lnl_batch(x[:period])

    def repeats(v):
        k = B // period * period
        assert torch.equal(v[:k].reshape(-1, period), v[:period].expand(k // period, period))
        assert torch.equal(v[k:], v[:B - k])

    lnl = m.lnl_batch(x)
    repeats(lnl)
    assert torch.allclose(lnl[:period], few, rtol=1e-12, atol=0)
    for which in ("single_pass", "two_pass"):
        m.set_grad_kernel(which)
        lnl, g = m.lnl_grad_batch(x)
        repeats(lnl)
        repeats(g[:, 0])
        assert torch.allclose(lnl[:period], few, rtol=1e-12, atol=0)
        assert torch.allclose(g[:period, 0], m.lnl_grad_batch(x[:period])[1][:, 0], rtol=1e-9, atol=1e-9)
    assert m.nonfinite_count() == 0
