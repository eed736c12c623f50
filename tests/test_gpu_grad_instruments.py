"""The single-pass adjoint keeps its per-instrument and acceleration sums in LDS
in up to eight copies, fewer with many instruments or MA sets: instruments 1 to
16, with the MA absent, global or per instrument, timescales fixed and free, an
acceleration, and multipliers near one (every tile then leaves R states behind).
Against the two-pass kernel, which computes the same sums in another order: lnL
to 1e-12 relative and the gradient to 1e-9 of max(|g|, 1), the bounds the two
kernels are held to on the catalogue stars."""
import numpy as np
import pytest

from astroemperor_amd import (AccelerationBlock, JitterBlock, KeplerianBlock, MOAVBlock, OffsetBlock, ReddModel, RVData,
                              SmartSetter)

pytestmark = pytest.mark.gpu


def _model(I, ma, free, strong, acc, rng):
    n = 41
    span = 40.0 if strong else 3000.0
    bjd = [np.sort(2450000.0 + rng.uniform(0, span, n + 3 * i)) for i in range(I)]
    data = RVData.from_arrays(bjd, [rng.normal(0, 5, len(b)) for b in bjd], [rng.uniform(1, 3, len(b)) for b in bjd])
    blocks = [KeplerianBlock(1, 1)] + ([AccelerationBlock(acc)] if acc else []) + [OffsetBlock(I), JitterBlock(I)]
    if ma:
        blocks.append(MOAVBlock(I, {"order": 1, "global": ma == "global"}))
    ss = SmartSetter(data.as_table())
    for b in blocks:
        ss(b)
        for p in b:
            if p.name.startswith("MACoefficient"):
                p.limits = [0.9, 0.99] if strong else [-0.5, 0.5]
            if p.name.startswith("MATimescale") and not free:
                p.fixed = 5.0
            if p.name.startswith("Period"):
                p.limits = [2.0, 900.0]
            if p.name.startswith("Amplitude"):
                p.limits = [1.0, 20.0]
            if p.name.startswith("Offset"):
                p.limits = [-20.0, 20.0]
            if p.name.startswith("Jitter"):
                p.limits = [0.1, 5.0]
            if p.name.startswith("Acceleration"):
                p.limits = [-0.01, 0.01]
    return ReddModel(blocks, data, semantics="intended")


@pytest.mark.parametrize("I,ma,free,strong,acc", [
    (1, None, False, False, 2), (16, None, False, False, 0), (1, "global", False, False, 1), (5, "instrument", False, False, 0),
    (8, "global", True, True, 0), (16, "global", False, True, 2), (9, "instrument", True, False, 1),
    (16, "instrument", True, True, 4)])
def test_copies_of_the_sums(I, ma, free, strong, acc):
    rng = np.random.default_rng(1000 + 10 * I + acc)
    m = _model(I, ma, free, strong, acc, rng)
    lim = m.limits_free()
    th = lim[:, 0] + (lim[:, 1] - lim[:, 0]) * rng.uniform(0.05, 0.95, size=(33, len(lim)))
    for j, nm in enumerate(m.names_free()):
        if nm.startswith("Ecc_sin"):
            th[:, j:j + 2] *= 0.65
    for prec in ("fp64", "mixed"):
        m.set_grad_kernel("two_pass")
        l0, g0 = m.lnl_grad_batch(th, prec)
        m.set_grad_kernel("auto")
        l1, g1 = m.lnl_grad_batch(th, prec)
        assert np.all(np.isfinite(l0))
        assert np.all(np.abs(l1 - l0) <= 1e-12 * np.abs(l0))
        assert np.all(np.abs(g1 - g0) <= 1e-9 * np.maximum(np.abs(g0), 1.0))
