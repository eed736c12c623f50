"""The mixed path's planet term for series of 64 to 255 epochs, where it solves
Kepler's equation to FP64 accuracy.  One epoch carries almost all of the weight, so
that the difference of the mixed and the FP64 lnL is that epoch's difference of the
term, d = dlnL sigma^2 / r.

Tolerance.  Both paths reduce the same bits of M.  E is rounded to 4.4e-16 (E up to
pi) on each side, which the term's slope in E, at most that in M,
K sqrt((1 + e) / (1 - e)^3), carries over; the term is at most (1 + e) K and takes a
handful of roundings; lnL itself is rounded to a few 1.1e-16 of r^2 / 2 sigma^2, with
r up to 4 K, some 1e-15 K of d.  A start whose error reached the result would show:
Newton's step leaves 6e-14 rad at e = 0.5, Halley's from 3.5e-5 rad 1.5e-14."""
import numpy as np
import pytest

from astroemperor_amd import KeplerianBlock, OffsetBlock, ReddModel, RVData, SmartSetter

pytestmark = pytest.mark.gpu


def errors(n, lo, hi, wpt, B=2000, K=10.0):
    rng = np.random.default_rng(int(1000 * hi) + n)
    t = 2450000.0 + np.sort(rng.uniform(0.0, 3000.0, n))
    sig = np.full(n, 1e7)
    sig[n // 2] = 1e-3
    data = RVData.from_arrays([t], [rng.normal(size=n)], [sig])
    kb, ob = KeplerianBlock(0, 1), OffsetBlock(1)
    ss = SmartSetter(data.as_table())
    ss(kb)
    ss(ob)
    m = ReddModel([kb, ob], data)
    m.set_waves_per_theta(wpt)
    e = rng.uniform(lo, hi, B)
    e[0] = hi
    th = np.stack([rng.uniform(3000.0, 9000.0, B), np.full(B, K), rng.uniform(0, 2 * np.pi, B), e,
                   rng.uniform(0, 2 * np.pi, B), np.full(B, 2 * K)], axis=1)
    mu = np.array([m.my_model(x)[0][n // 2] for x in th])
    r = m.data.Y[n // 2] - mu
    d = []
    for f in (m.lnl_batch, lambda x, p: m.lnl_grad_batch(x, p)[0]):
        d.append((f(th, "mixed") - f(th, "fp64")) * 1e-6 / r)
    tol = K * (4e-15 + 1e-15 * np.sqrt((1 + e) / (1 - e) ** 3))
    return np.abs(np.array(d)), np.where(np.abs(r) > 0.5 * K, tol, np.inf), K


@pytest.mark.parametrize("wpt", [1, 4])
@pytest.mark.parametrize("n", [64, 200, 255])
@pytest.mark.parametrize("lo,hi", [(0.0, 0.5), (0.5, 0.75), (0.75, 0.95)])
def test_term_to_fp64_accuracy(lo, hi, n, wpt):
    d, tol, K = errors(n, lo, hi, wpt)
    print(f"e {lo}-{hi} n {n} wpt {wpt}: max {d[:, np.isfinite(tol)].max() / K:.1e} K, "
          f"rms {np.sqrt(np.mean(d[:, np.isfinite(tol)] ** 2)) / K:.1e} K")
    assert np.isfinite(tol).mean() > 0.7
    assert np.all(d <= tol)
