"""Batched skies over a segment of more antenna frames than 64 times 65,536
(needs a GPU): the occlusion bits' launch covers them all.  Weights equal the
one-sky form's, maps to the mixed bar."""
import numpy as np
import pytest

from _lockstep import MIXED_TOL, config, rel_err
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu


def test_many_frames():
    n = 2097200  # 4,194,400 frames of two antennas; 65,536 x 64 = 4,194,304
    kw = dict(nside=2, n_ant=2, n_epochs=n, segs=1, img_n=0, freq_hz=1e6, dt_s=1.0)
    skies = np.random.default_rng(9).lognormal(0.0, 1.0, (2, 48))
    with Pipeline(config(precision=1, nsky=2, **kw)) as b:
        b.set_sky(skies)
        b.run_all()
        C, W, _, _ = b.finalize()
        for s in range(2):
            with Pipeline(config(**kw)) as p:
                p.set_sky(skies[s])
                p.run_all()
                Cp, Wp, _, _ = p.finalize()
            assert np.array_equal(W, Wp)
            assert rel_err(C[s], Cp) <= MIXED_TOL
