"""The gradient move's preconditioner over its instances: parameter counts in one
to seven 16-column tiles (matrix instructions, panels of four columns with a
remainder), walker counts that are no multiple of the waves' share, and a
parameter without spread.  One sweep of gradient moves from walkers around a
point (spread 1e-7 of the prior's width, so that the move accepts) is replayed on
the host as in the replay test of the two moves.  Positions to 1e-6 of the
spread: a position's rounding is 2e-9 of it, which the factor of a covariance of
condition number about 30 and the gradients (1e-9) carry to some 1e-7."""
import numpy as np
import pytest

from tests.conftest import make_sim, oracle_for
from tests.test_gpu_moves import _PostG, _replay

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,moav,acc,W", [(1, None, 0, 34), (2, None, 1, 62), (5, None, 0, 110), (7, None, 0, 158),
                                          (8, {"order": 3, "global": False}, 0, 206), (0, None, 0, 10)])
def test_one_sweep_replays(k, moav, acc, W):
    from astroemperor_amd import GradientMove, PTSampler
    sim = make_sim("GJ876", k, parameterisation=1, moav=moav, acceleration=acc, semantics="intended")
    m = sim.model
    D = m.ndim__
    rng = np.random.default_rng(40 + k)
    lim = m.limits_free()
    mid = lim[:, 0] + 0.4 * (lim[:, 1] - lim[:, 0])
    for j, nm in enumerate(m.names_free()):
        if nm.startswith("Ecc_"):
            mid[j] = 0.2
    T, seed, eps = 2, 99 + k, 0.05
    betas = np.array([1.0, 0.2])
    width = 1e-7 * (lim[:, 1] - lim[:, 0])
    X = mid + width * rng.normal(size=(T, W, D))
    X[1, :, D // 2] = np.float32(mid[D // 2])            # no spread: does not move
    s = PTSampler(W, D, m, ntemps=T, betas=betas, adapt_mode=-1, seed=seed, moves=[(GradientMove(eps), 1.0)])
    s.run_mcmc(X.copy(), nsweeps=1, capacity=1)
    o = oracle_for(m)
    lnl = np.array([[o.my_likelihood(x) for x in X[t]] for t in range(T)])
    lnp = np.array([[o.my_prior(x) for x in X[t]] for t in range(T)])
    X0 = X.copy()
    acc_ = _replay(o, _PostG(o, m), X, lnl, lnp, betas, 0, seed, 1, eps)
    got = s.get_last_sample()
    assert np.all(np.abs(got.coords - X) <= 1e-6 * width)
    assert np.array_equal(s._get(6, np.int64)[..., 0, 0], acc_)
    assert acc_.sum() > 0 and (X != X0).any()
