"""The deconvolver's FP16 kernels at image sides whose levels are no multiples
of eight (rows on any two bytes, tails of 1 to 7 pixels, tiles cut by the
image), against the FP16 oracle.  Outputs to 5e-3 of the largest as in
test_gpu_unet.  With 1 to 121 pixels at the deepest level a pre-activation that
rounds to the other side of zero moves single weight gradients by its pixel's
whole share, so gradients are held per layer in the 2-norm: a share of 1 / 27 in
one of 27 pixels' terms stays below 5e-2, a dropped or doubled row tail does not."""
import numpy as np
import pytest

import test_gpu_unet as T
from oracle import unet_ref as U
from viss_optimize_ws_amd.deconv import UNet

pytestmark = pytest.mark.gpu


# sides by level: 24 12 6 3 | 40 20 10 5 | 56 28 14 7 | 72 36 18 9 | 88 44 22 11
@pytest.mark.parametrize("N,n", [(24, 3), (40, 2), (56, 2), (72, 2), (88, 1)])
def test_ragged_levels(N, n):
    rng = np.random.default_rng(21)
    x, y = (rng.normal(size=(n, N, N)).astype(np.float32) for _ in range(2))
    with UNet(N, n, fp16=True, seed=1) as net:
        net.set_params(T._params(22).astype(np.float32))
        th = net.params().astype(np.float64)
        out = net.predict(x)
        loss, g = net.loss_grad(x, y)
    ref, _ = U.forward(th, x, fp16=True)
    lref, gref = U.loss_grad(th, x, y, fp16=True)
    assert np.max(np.abs(out - ref)) <= 5e-3 * np.max(np.abs(ref))
    assert abs(loss - lref) <= 5e-3 * lref
    off = 0
    for k, (ci, co, _) in enumerate(U.SPEC):
        m = co * ci * (9 if k < 14 else 1) + co
        d, r = g[off:off + m] - gref[off:off + m], gref[off:off + m]
        assert np.linalg.norm(d) <= 5e-2 * np.linalg.norm(r), (k, np.linalg.norm(d) / np.linalg.norm(r))
        off += m
