"""Engines on one device read with another device current: the getters' gather
buffer belongs to the engine's device, and the caller's device stays current."""
import numpy as np
import pytest
import torch

from tests.conftest import make_sim

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two devices")]


def test_state_read_from_another_device():
    from astroemperor_amd import PTSampler, SystemsPT
    from astroemperor_amd.simulation import test_init
    rng = np.random.default_rng(1)
    with torch.cuda.device(1):
        m = make_sim("51Peg", 1, parameterisation=1).model
        p0 = test_init(m, 2, 16, rng)
        s = PTSampler(16, m.ndim__, m, ntemps=2, seed=3)
        here = s.run_mcmc(p0, nsweeps=4)
        y = SystemsPT([m], 2, 16, [p0], seed=3)
        y.run(4)
        x1, l1, _ = y.state(0)
        mean = s.lnl_moments(1)[0]
    with torch.cuda.device(0):
        there = s.get_last_sample()
        assert np.array_equal(here.coords, there.coords) and np.array_equal(here.log_like, there.log_like)
        x0, l0, _ = y.state(0)
        assert np.array_equal(x0, x1) and np.array_equal(l0, l1)
        assert np.array_equal(s.lnl_moments(1)[0], mean)
        assert torch.cuda.current_device() == 0
