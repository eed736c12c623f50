"""Switching the adjoint kernel under an enabled gradient move."""
import numpy as np
import pytest

from tests.conftest import make_sim

pytestmark = pytest.mark.gpu


def test_two_pass_after_the_gradient_move_short_series():
    """Below 1024 epochs the gradient move holds the eps rows of the two-pass
    adjoint although the default does not use them: the kernel may be switched
    after the move was enabled, and both sample the same chain to rounding."""
    from astroemperor_amd import GradientMove, PTSampler
    ends = []
    for which in ("auto", "two_pass"):
        sim = make_sim("GJ876", 1, parameterisation=1, moav={"order": 1, "global": False}, semantics="intended")
        m = sim.model
        lim = m.limits_free()
        rng = np.random.default_rng(7)
        p0 = lim[:, 0] + (lim[:, 1] - lim[:, 0]) * rng.uniform(0.3, 0.6, size=(2, 32, len(lim)))
        s = PTSampler(32, m.ndim__, m, ntemps=2, seed=5, moves=[GradientMove(1e-3)])
        s.run_mcmc(p0, nsweeps=1, capacity=4)
        m.set_grad_kernel(which)
        ends.append(s.run_mcmc(None, nsweeps=3).log_like)
    assert np.allclose(ends[0], ends[1], rtol=1e-8, atol=1e-6)
