"""The gradient move's preconditioner on both sides of every change of its
instance (16, 32, 48, 64 and 96 parameters; column tiles 1, 2, 3, 4, 6, 8), and
inside the widest ones.  One sweep of gradient moves is replayed on the host as
in the replay test of the two moves, and two runs from one seed are the same
bits: the factor is a function of the positions alone.  Walkers have a spread of
1e-7 of the prior's width around a point, so that the move accepts.  Positions to
1e-6 of the spread: a position's rounding is 2e-9 of it, which the factor of a
covariance of condition number (1 + r)^2 / (1 - r)^2, r^2 = D / (W / 2) <= 2/3, of
at most 98 and the gradients (1e-9) carry to some 2e-7."""
import numpy as np
import pytest

from astroemperor_amd import (GradientMove, JitterBlock, KeplerianBlock, MagneticCycleBlock, MOAVBlock, OffsetBlock,
                              PTSampler, ReddModel, RVData, SinusoidBlock, SmartSetter)
from tests.conftest import oracle_for
from tests.test_gpu_moves import _PostG, _replay

pytestmark = pytest.mark.gpu

# planets, MA order (0: none), sinusoid, magnetic cycle, offsets held fixed; parameters, column tiles
CASES = [((0, 0, 0, 0, 0), 16, 1), ((1, 0, 0, 0, 4), 17, 2), ((4, 0, 0, 0, 4), 32, 2), ((4, 0, 0, 0, 3), 33, 3),
         ((7, 0, 0, 0, 3), 48, 3), ((7, 0, 0, 0, 2), 49, 4), ((7, 1, 0, 0, 3), 64, 4), ((7, 1, 0, 0, 2), 65, 6),
         ((7, 1, 0, 0, 0), 67, 6), ((7, 2, 0, 0, 0), 83, 6), ((8, 2, 1, 1, 0), 96, 6), ((8, 3, 0, 0, 7), 97, 8)]


def _instance(D):
    return next(n for n in (1, 2, 3, 4, 6, 8) if D <= 16 * n)


def _model(k, q, sin, mag, nfix):
    """A small star of eight instruments."""
    rng = np.random.default_rng(17 * k + q)
    I = 8
    bjd = [np.sort(2450000.0 + rng.uniform(0.0, 1000.0, 9)) for _ in range(I)]
    data = RVData.from_arrays(bjd, [rng.normal(0.0, 5.0, 9) for _ in bjd], [rng.uniform(1.0, 3.0, 9) for _ in bjd])
    blocks = [KeplerianBlock(1, p + 1) for p in range(k)]
    blocks += [OffsetBlock(I), JitterBlock(I)]
    blocks += [MOAVBlock(I, {"order": q, "global": False})] if q else []
    blocks += [SinusoidBlock(1)] if sin else []
    blocks += [MagneticCycleBlock(1)] if mag else []
    ss = SmartSetter(data.as_table())
    for b in blocks:
        ss(b)
        for p in list(b)[:nfix] if b.type_ == "Offset" else ():
            p.fixed = 0.5
    return ReddModel(blocks, data, semantics="intended")


def test_cases_reach_every_instance():
    assert all(_instance(D) == n for _, D, n in CASES)
    assert {n for _, _, n in CASES} == {1, 2, 3, 4, 6, 8}


@pytest.mark.parametrize("spec,D,tiles", CASES)
def test_one_sweep_replays_and_repeats(spec, D, tiles):
    m = _model(*spec)
    assert m.ndim__ == D
    rng = np.random.default_rng(D)
    lim = m.limits_free()
    mid = lim[:, 0] + 0.4 * (lim[:, 1] - lim[:, 0])
    for j, nm in enumerate(m.names_free()):
        if nm.startswith("Ecc_"):
            mid[j] = 0.2
    T, W, seed, eps = 1, 3 * D + 3 + (D + 1) % 2, 500 + D, 0.05
    betas = np.array([1.0])
    width = 1e-7 * (lim[:, 1] - lim[:, 0])
    X = mid + width * rng.normal(size=(T, W, D))
    X[0, :, -1] = np.float32(mid[-1])                 # no spread: does not move
    runs = []
    for _ in range(2):
        s = PTSampler(W, D, m, ntemps=T, betas=betas, adapt_mode=-1, seed=seed, moves=[(GradientMove(eps), 1.0)])
        s.run_mcmc(X.copy(), nsweeps=1, capacity=1)
        runs.append((s.get_last_sample(), s._get(6, np.int64)[..., 0, 0]))
        s.close()
    assert np.array_equal(runs[0][0].coords, runs[1][0].coords)
    assert np.array_equal(runs[0][0].log_like, runs[1][0].log_like)
    assert np.all(runs[0][0].coords[0, :, -1] == X[0, 0, -1])
    o = oracle_for(m)
    lnl = np.array([[o.my_likelihood(x) for x in X[t]] for t in range(T)])
    lnp = np.array([[o.my_prior(x) for x in X[t]] for t in range(T)])
    X0 = X.copy()
    acc = _replay(o, _PostG(o, m), X, lnl, lnp, betas, 0, seed, 1, eps)
    got, accepted = runs[0]
    assert np.all(np.abs(got.coords - X) <= 1e-6 * width)
    assert np.array_equal(accepted, acc)
    assert acc.sum() > 0 and (X != X0).any()
