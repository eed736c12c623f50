"""The batched prior evaluates the terms of 16 vectors by the lanes of a workgroup
and adds each vector's up in order, eight at a time.  Short and long sequences,
batches that are not a multiple of the workgroup's vectors, padded rows, and
vectors outside their support, against the oracle: the terms are those of the
oracle to an ulp and each of the n additions rounds once, so n ulps of the
(one-signed) sum; a row's prior doesn't depend on its batch."""
import numpy as np
import pytest
import torch

from tests.conftest import make_sim, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,moav,acc", [(0, None, 0), (1, None, 1), (5, {"order": 1, "global": False}, 0),
                                        (7, {"order": 3, "global": False}, 2)])
def test_prior_terms_against_oracle(k, moav, acc):
    sim = make_sim("GJ876", k, parameterisation=1, moav=moav, acceleration=acc, semantics="intended")
    m = sim.model
    rng = np.random.default_rng(100 + k)
    lim = m.limits_free()
    D = len(lim)
    th = lim[:, 0] + (lim[:, 1] - lim[:, 0]) * rng.uniform(size=(131, D))
    for q, nm in enumerate(m.names_free()):
        if nm.startswith("Ecc_sin"):
            th[:, q:q + 2] *= 0.5
    for r in range(0, 131, 5):
        th[r, rng.integers(D)] = [np.inf, -np.inf, np.nan, lim[:, 1].max() * 10 + 1][r % 4]
    o = oracle_for(m)
    ref = np.array([o.my_prior(t) for t in th])
    got = m.lnprior_batch(th)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isfinite(got), fin) and fin.sum() > 40 and (~fin).sum() > 5
    assert np.all(np.abs(got[fin] - ref[fin]) <= (D + k) * np.spacing(np.abs(ref[fin])))
    pad = torch.full((131, D + 3), float("nan"), dtype=torch.float64, device="cuda")
    pad[:, :D] = torch.from_numpy(th).cuda()
    for b in (1, 15, 16, 17, 130):
        assert np.array_equal(m.lnprior_batch(th[:b]), got[:b])
        assert np.array_equal(m.lnprior_batch(pad[:b, :D]).cpu().numpy(), got[:b])
