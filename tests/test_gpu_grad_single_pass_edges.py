"""The single-pass adjoint at the sizes where its layout can go wrong: series
shorter than a wave's pairs, around one and two 256-epoch tiles, odd lengths
(a lane with one epoch), and planet counts on both sides of the register
instances (4, 6, 8), without the moving average, with it per instrument
(epochs grouped) and globally (instruments interleaved), and with multipliers
near one (every wave of a tile then carries its A parts).  The two-pass kernel
computes the same sums in another order: lnL to 1e-12 relative and the
gradient to 1e-9 of max(|g|, 1), the bounds the two kernels are held to on the
catalogue stars."""
import numpy as np
import pytest

from astroemperor_amd import (AccelerationBlock, JitterBlock, KeplerianBlock, MOAVBlock, OffsetBlock, ReddModel, RVData,
                              SmartSetter)

pytestmark = pytest.mark.gpu


def _model(n, k, ma, rng, param, acc=0):
    counts = [max(1, n // 2), max(1, n // 3)]
    counts.append(max(1, n - sum(counts)))
    n = sum(counts)
    bjd = [np.sort(2450000.0 + rng.uniform(0, 40.0 if ma == "strong" else 3000.0, c)) for c in counts]
    data = RVData.from_arrays(bjd, [rng.normal(0, 5, c) for c in counts], [rng.uniform(1, 3, c) for c in counts])
    blocks = [KeplerianBlock(param, q + 1) for q in range(k)]
    if acc:
        blocks.append(AccelerationBlock(acc))
    blocks += [OffsetBlock(3), JitterBlock(3)]
    if ma != "none":
        blocks.append(MOAVBlock(3, {"order": 1, "global": ma == "global"}))
    ss = SmartSetter(data.as_table())
    for b in blocks:
        ss(b)
        for p in b:
            if p.name.startswith("MACoefficient"):
                p.limits = [0.9, 0.99] if ma == "strong" else [-0.5, 0.5]
            if p.name.startswith("MATimescale") and ma == "instrument":
                p.fixed = 5.0
            if p.name.startswith(("Period", "lPeriod")):
                p.limits = [np.log(2.0), np.log(900.0)] if p.name.startswith("l") else [2.0, 900.0]
            if p.name.startswith("Amplitude"):
                p.limits = [1.0, 20.0]
            if p.name.startswith("Offset"):
                p.limits = [-20.0, 20.0]
            if p.name.startswith("Jitter"):
                p.limits = [0.1, 5.0]
    return ReddModel(blocks, data, semantics="intended")


def _draws(m, n, rng):
    lim = m.limits_free()
    th = lim[:, 0] + (lim[:, 1] - lim[:, 0]) * rng.uniform(0.05, 0.95, size=(n, len(lim)))
    names = m.names_free()
    for j, nm in enumerate(names):
        if nm.startswith("Ecc_sin"):
            th[:, j:j + 2] *= 0.65
        if nm.startswith("Eccentricity"):
            th[:, j] *= 0.95
    return th


@pytest.mark.parametrize("ma", ["none", "instrument", "global", "strong"])
@pytest.mark.parametrize("n,k,param,acc", [(3, 1, 1, 0), (63, 2, 6, 0), (128, 4, 1, 1), (255, 5, 6, 0), (256, 6, 1, 0),
                                           (257, 7, 6, 2), (511, 8, 3, 0), (513, 3, 0, 0), (1025, 4, 4, 0)])
def test_matches_two_pass(n, k, param, acc, ma):
    rng = np.random.default_rng(n * 10 + k)
    m = _model(n, k, ma, rng, param, acc)
    th = _draws(m, 5, rng)
    for p in ("fp64", "mixed"):
        m.set_grad_kernel("two_pass")
        l2, g2 = m.lnl_grad_batch(th, p)
        m.set_grad_kernel("single_pass")
        l1, g1 = m.lnl_grad_batch(th, p)
        m.set_grad_kernel("auto")
        l0, g0 = m.lnl_grad_batch(th, p)
        assert np.array_equal(l0, l1) and np.array_equal(g0, g1)          # the default is the single-pass kernel
        assert np.isfinite(l2).all()
        assert np.max(np.abs(l1 - l2) / np.abs(l2)) < 1e-12
        assert np.max(np.abs(g1 - g2) / np.maximum(np.abs(g2), 1.0)) < 1e-9
