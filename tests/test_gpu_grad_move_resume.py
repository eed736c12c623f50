"""A run with gradient moves and a moving average resumes bitwise at an ensemble
whose current positions and whose proposals are batches on different sides of the
adjoint's change of shape (three vectors per compute unit): a restored engine
recomputes every gradient in one launch over the positions, the other kept those
of the accepted proposals, and both must be the same bits."""
import numpy as np
import pytest

from astroemperor_amd import GradientMove, PTSampler, device_info
from tests.conftest import make_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ma", [False, True])          # per instrument, global
def test_resumes_bitwise_across_the_shapes(tmp_path, ma):
    m = make_sim("GJ876", 0, moav={"order": 1, "global": ma}, semantics="intended").model
    T, W = 4, int(device_info()["n_cu"])                # 4 walkers per compute unit, 2 proposals
    rng = np.random.default_rng(8)
    lim = m.limits_free()
    start = [(0.0, 15.0) if n.startswith("Offset") else (150.0, 10.0) if n.startswith("Jitter") else
             (0.1, 0.05) if n.startswith("MACoefficient") else (6.0, 0.5) for n in m.names_free()]
    p0 = np.clip([[[rng.normal(*q) for q in start] for _ in range(W)] for _ in range(T)],
                 lim[:, 0] + 1e-6, lim[:, 1] - 1e-6)
    moves = [(GradientMove(0.5), 1.0)]
    s = PTSampler(W, m.ndim__, m, ntemps=T, seed=11, moves=moves)
    s.run_mcmc(p0, nsweeps=8, capacity=16)
    s.checkpoint(tmp_path / "ck.bin")
    s.run_mcmc(None, nsweeps=8)
    s2 = PTSampler(W, m.ndim__, m, ntemps=T, seed=11, moves=moves)
    s2.run_mcmc(p0, nsweeps=0, capacity=16)
    s2.restore(tmp_path / "ck.bin")
    s2.run_mcmc(None, nsweeps=8)
    assert s.accepted.mean() > 1.0                      # gradient proposals are accepted
    assert np.array_equal(s.get_chain(), s2.get_chain())
    assert np.array_equal(s.get_log_like(), s2.get_log_like())
