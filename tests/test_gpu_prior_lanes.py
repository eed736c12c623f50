"""The batched prior's three kernels (16 vectors per workgroup; a lane per vector with
whole rows in LDS, up to 24 parameters; a lane per vector with 16 terms at a time)
form the same bits: batches on both sides of the change of kernel (a wave per SIMD,
two for long rows), with remainders, padded rows, vectors outside their support and
values that are no numbers, against the same vectors in small batches."""
import numpy as np
import pytest
import torch

from astroemperor_amd import (JitterBlock, KeplerianBlock, MOAVBlock, OffsetBlock, ReddModel, RVData, SmartSetter,
                              device_info)

pytestmark = pytest.mark.gpu


def _model(k, I, q, param):
    rng = np.random.default_rng(k)
    bjd = [np.sort(2450000.0 + rng.uniform(0.0, 1000.0, 6)) for _ in range(I)]
    data = RVData.from_arrays(bjd, [rng.normal(0.0, 5.0, 6) for _ in bjd], [rng.uniform(1.0, 3.0, 6) for _ in bjd])
    blocks = [KeplerianBlock(param, p + 1) for p in range(k)] + [OffsetBlock(I)]
    blocks += [JitterBlock(I)] if k else []
    blocks += [MOAVBlock(I, {"order": q, "global": False})] if q else []
    ss = SmartSetter(data.as_table())
    for b in blocks:
        ss(b)
    return ReddModel(blocks, data, semantics="intended")


@pytest.mark.parametrize("k,I,q,param,D", [(0, 1, 0, 1, 1), (1, 1, 0, 1, 7), (4, 2, 0, 6, 24), (3, 5, 0, 1, 25),
                                           (7, 8, 1, 1, 67), (8, 8, 3, 0, 104)])
def test_same_bits_as_small_batches(k, I, q, param, D):
    m = _model(k, I, q, param)
    assert m.ndim__ == D
    rng = np.random.default_rng(D)
    lim = m.limits_free()
    n = 4001
    th = lim[:, 0] + (lim[:, 1] - lim[:, 0]) * rng.uniform(size=(n, D))
    for j, nm in enumerate(m.names_free()):
        if nm.startswith("Ecc_sin"):
            th[:, j:j + 2] *= 0.6
    for r in range(0, n, 5):
        th[r, rng.integers(D)] = [np.inf, -np.inf, np.nan, lim[:, 1].max() * 10 + 1, lim[0, 0]][r // 5 % 5]
    ref = torch.from_numpy(m.lnprior_batch(th)).cuda()
    assert torch.isfinite(ref).sum() > n // 3 and (~torch.isfinite(ref)).sum() > n // 10
    most = 256 * int(device_info()["n_cu"]) * (1 if D <= 24 else 2)
    rows = torch.from_numpy(th).cuda()[torch.arange(most + 65, device="cuda") % n]
    want = ref[torch.arange(most + 65, device="cuda") % n]
    pad = torch.full((most + 65, D + 3), float("nan"), dtype=torch.float64, device="cuda")
    pad[:, :D] = rows
    for B in (most - 1, most, most + 1, most + 63, most + 65):
        for x in (rows[:B], pad[:B, :D]):
            assert torch.equal(torch.nan_to_num(m.lnprior_batch(x), nan=7.0), torch.nan_to_num(want[:B], nan=7.0)), B
