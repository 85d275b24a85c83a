"""Device memory of contexts with large maps and short segments (needs a GPU)."""
import numpy as np
import pytest

from _lockstep import config, rel_err
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu


def test_large_map_partials():
    """Nside 1024, segments of a few rows.  A pixel holds its direction (32 bytes), sky (12), accumulators and outputs
    (24) and the partial sum and count of one group range (12): 80 bytes, with a third as much for tiles and tables.
    Ranges for every segment of a merged run, or for as many as a run could have, would take 12 bytes each.  The maps of
    a step and of the stage calls are those of the same sums."""
    cfg = dict(nside=1024, n_ant=3, n_epochs=9, segs=3, img_n=0, freq_hz=1e7)
    with Pipeline(config(**cfg)) as p:
        assert p.plan.device_bytes <= 107 * p.plan.npix, p.plan.device_bytes / p.plan.npix
        p.set_sky(np.random.default_rng(1).lognormal(0.0, 1.0, p.plan.npix))
        p.run_all()
        C, W, _, _ = p.finalize()
        p.reset_accumulators()
        for t0, tl in p.schedule():
            p.gen_segment(t0, tl)
            p.viss_half()
            p.conj_fill()
            p.recon_segment()
        C2, W2, _, _ = p.finalize()
    assert np.array_equal(W, W2) and rel_err(C, C2) <= 1e-10
