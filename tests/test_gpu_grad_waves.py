"""The single-pass adjoint's shapes: one wave per vector up to 128 epochs; with a
moving average four (tiles of 512 epochs) up to three vectors per compute unit of
more than 256 epochs; else two (tiles of 256).  On both sides of these limits and
around one and two tiles, against the two-pass kernel, which computes the same sums
in another order: lnL to 1e-12 relative and the gradient to 1e-9 of max(|g|, 1), the
bounds the two kernels are held to on the catalogue stars."""
import numpy as np
import pytest

from astroemperor_amd import device_info
from tests.test_gpu_grad_single_pass_edges import _draws, _model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ma", ["none", "instrument", "global", "strong"])
@pytest.mark.parametrize("n,k,param,acc", [(7, 1, 1, 0), (127, 8, 6, 0), (128, 5, 1, 0), (129, 7, 6, 2), (255, 2, 6, 0), (256, 4, 1, 1), (257, 6, 1, 0), (511, 8, 3, 0),
                                           (512, 7, 6, 0), (513, 3, 0, 2), (1023, 5, 6, 0), (1025, 4, 4, 0)])
def test_both_shapes_match_two_pass(n, k, param, acc, ma):
    rng = np.random.default_rng(n + k)
    m = _model(n, k, ma, rng, param, acc)
    most = 3 * int(device_info()["n_cu"])
    th = _draws(m, most + 1, rng)
    for p in ("fp64", "mixed"):
        m.set_grad_kernel("two_pass")
        l2, g2 = m.lnl_grad_batch(th, p)
        m.set_grad_kernel("single_pass")
        assert np.isfinite(l2).all()
        for B in (1, 3, most, most + 1):
            l1, g1 = m.lnl_grad_batch(th[:B], p)
            assert np.max(np.abs(l1 - l2[:B]) / np.abs(l2[:B])) < 1e-12
            assert np.max(np.abs(g1 - g2[:B]) / np.maximum(np.abs(g2[:B]), 1.0)) < 1e-9
