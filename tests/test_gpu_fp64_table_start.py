"""FP64 Kepler solve from the per-vector table start (planet_sc with PREC 0)
against the oracle, in every eccentricity band that takes another step, at
both forms of the table and around the shortest series that has one.

Tolerance.  Periods of at least the time span keep M = 2 pi t / P + M0 below
4 pi, where one rounding is 8.9e-16; both sides round M, the products and the
angles a few times, so |dM| <= 4 x 8.9e-16, which moves a planet's term by at
most |dM| K sqrt((1 + e) / (1 - e)^3), the largest slope of K cos(f + w) in M.
Rounding of the term itself adds a few 1e-16 K.  A start whose error reached
the result would show: the coarsest step left out (the cubic term at
0.5 < e <= 0.75) is 2e-14 rad, the next ones 1e-13 and more.
"""
import numpy as np
import pytest

from astroemperor_amd import KeplerianBlock, OffsetBlock, ReddModel, RVData, SmartSetter
from oracle.emp_oracle import OracleModel

pytestmark = pytest.mark.gpu
EPS = 8.9e-16
BANDS = [(0.0, 0.3), (0.3, 0.5), (0.5, 0.75), (0.75, 0.95), (0.95, 0.98)]


def _star(n, rng):
    t = np.sort(rng.uniform(0.0, 3000.0, n))
    t[0] = 0.0
    data = RVData.from_arrays([2450000.0 + t], [rng.normal(size=n)], [rng.uniform(1.0, 2.0, n)])
    ss = SmartSetter(data.as_table())
    kb, ob = KeplerianBlock(0, 1), OffsetBlock(1)
    ss(kb)
    ss(ob)
    return ReddModel([kb, ob], data)


@pytest.mark.parametrize("n", [255, 256, 700])
@pytest.mark.parametrize("lo,hi", BANDS)
def test_fp64_bands_vs_oracle(lo, hi, n):
    rng = np.random.default_rng(int(1000 * hi) + n)
    m = _star(n, rng)
    o = OracleModel(m.spec(), m.data.X, m.data.Y, m.data.YERR, m.data.FLAG)
    B, K = 24, 10.0
    e = rng.uniform(lo, hi, B)
    e[0] = hi                                   # the band's edge belongs to the lower step
    theta = np.stack([rng.uniform(3000.0, 9000.0, B), np.full(B, K), rng.uniform(0, 2 * np.pi, B), e,
                      rng.uniform(0, 2 * np.pi, B), np.zeros(B)], axis=1)
    tol = K * (4 * EPS * np.sqrt((1 + e) / (1 - e) ** 3) + 8 * EPS)
    mu = np.stack([o.my_model(th)[0] for th in theta])
    for b in range(4):                          # the interval form (one vector per workgroup)
        got, _ = m.my_model(theta[b])
        assert np.max(np.abs(got - mu[b])) <= tol[b]
    r = m.data.Y - mu
    ref = np.array([o.my_likelihood(th) for th in theta])
    bound = tol * np.sum(np.abs(r) / m.data.YERR ** 2, axis=1) + 4e-16 * n ** 0.5 * np.abs(ref)
    for wpt in (1, 4):                          # nodes and intervals
        m.set_waves_per_theta(wpt)
        assert np.all(np.abs(m.lnl_batch(theta) - ref) <= bound)
