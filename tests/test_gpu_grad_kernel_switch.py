"""The adjoint kernel switched under an engine that has captured its gradient
sweeps: the next run takes the new kernel, the same bits as sweeps launched without
a graph and other bits than the old kernel's (the two differ in rounding); on a
series below 1024 epochs, whose scratch is set aside with the move, and above, whose
scratch is allocated by the run."""
import numpy as np
import pytest

from astroemperor_amd import GradientMove, JitterBlock, MOAVBlock, OffsetBlock, PTSampler, ReddModel, RVData, SmartSetter

pytestmark = pytest.mark.gpu


def _star(n):
    rng = np.random.default_rng(n)
    bjd = [np.sort(2450000.0 + rng.uniform(0.0, 3000.0, n // 2)) for _ in range(2)]
    data = RVData.from_arrays(bjd, [rng.normal(0.0, 5.0, n // 2) for _ in bjd], [np.full(n // 2, 2.0) for _ in bjd])
    blocks = [OffsetBlock(2), JitterBlock(2), MOAVBlock(2, {"order": 1, "global": False})]
    ss = SmartSetter(data.as_table())
    for b in blocks:
        ss(b)
    return ReddModel(blocks, data, semantics="intended")


def _run(n, switch, graph):
    m = _star(n)
    rng = np.random.default_rng(1)
    start = [(0.0, 0.3) if q.startswith("Offset") else (4.0, 0.2) if q.startswith("Jitter") else
             (0.1, 0.02) if q.startswith("MACoefficient") else (8.0, 0.5) for q in m.names_free()]
    p0 = np.array([[[rng.normal(*q) for q in start] for _ in range(32)] for _ in range(2)])
    s = PTSampler(32, m.ndim__, m, ntemps=2, seed=5, moves=[GradientMove(0.5)])
    s.run_mcmc(p0, nsweeps=3, capacity=9, use_graph=graph)
    for which in switch:
        m.set_grad_kernel(which)
        s.run_mcmc(None, nsweeps=3, use_graph=graph)
    assert s.accepted.sum() > 0
    return s.get_chain(), s.get_log_like()


@pytest.mark.parametrize("n", [300, 1100])
def test_captured_sweeps_follow_the_switch(n):
    keep, switched = ("auto", "auto"), ("two_pass", "single_pass")
    x0, l0 = _run(n, keep, True)
    x1, l1 = _run(n, switched, True)
    x2, l2 = _run(n, switched, False)
    assert np.array_equal(x1, x2) and np.array_equal(l1, l2)
    assert np.array_equal(x0[:, :3], x1[:, :3]) and not np.array_equal(x0, x1)
    assert np.allclose(l0, l1, rtol=1e-8, atol=1e-6)
