"""The plain form's automatic choice of the Viss sum where segments have few
epochs: the per-row sum's bits, or the antenna-factorized one's where that is
the faster (needs a GPU)."""
import numpy as np
import pytest

from _lockstep import config
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu


# one pass of the kernel; quads of epochs and blocks of antennas partly empty; their neighbours that gain by it
@pytest.mark.parametrize("nside,n_ant,n_epochs,form", [(16, 28, 1, 1), (32, 13, 7, 1), (32, 13, 8, 2), (32, 32, 2, 1),
                                                       (32, 32, 3, 2), (128, 22, 2, 1), (128, 32, 1, 2), (128, 13, 5, 1),
                                                       (128, 14, 8, 2), (256, 16, 2, 1), (256, 28, 3, 2)])
def test_form_by_epochs(nside, n_ant, n_epochs, form):
    v = []
    for f in (0, 1, 2):
        with Pipeline(config(nside=nside, n_ant=n_ant, n_epochs=n_epochs, segs=1, freq_hz=1e7, img_n=0, viss_form=f)) as p:
            p.set_sky(np.random.default_rng(n_ant).lognormal(0.0, 1.0, p.plan.npix))
            p.gen_segment(*p.schedule()[0])
            v.append(p.viss_half())
    assert not np.array_equal(v[1], v[2])
    assert np.array_equal(v[0], v[form])
