"""Whole steps whose Viss is far longer than their recon: the recon of a segment
runs beside the next one's Viss and does not hold it up, and the step gives what
one stream gives (needs a GPU)."""
import time

import numpy as np
import pytest

from _lockstep import MIXED_TOL, config, rel_err
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu


# both sides of the rule that puts the grouping after the Viss: pairs x points, epochs x pixels
@pytest.mark.parametrize("kw", [dict(nside=128, n_ant=8, n_epochs=190, segs=2), dict(nside=128, n_ant=8, n_epochs=160, segs=2),
                                dict(nside=128, n_ant=8, n_epochs=190, segs=2, img_n=30), dict(nside=64, n_ant=4, n_epochs=700, segs=2),
                                dict(nside=64, n_ant=5, n_epochs=700, segs=2, recon_mode=1, occ_mode=1),
                                dict(nside=64, n_ant=4, n_epochs=700, segs=2, blockage=0)])
def test_step_equals_one_stream(kw):
    base = dict(img_n=0, precision=1, freq_hz=1e7)
    base.update(kw)
    out = []
    for serial in (0, 1):
        with Pipeline(config(serial_stages=serial, **base)) as p:
            p.set_sky(np.random.default_rng(3).lognormal(0.0, 1.0, p.plan.npix))
            for _ in range(2):
                p.reset_accumulators()
                p.run_all()
            out.append(p.finalize())
    for a, b in zip(*out):
        if a is not None:
            assert np.array_equal(a, b) if a.dtype == np.uint32 else rel_err(a, b) <= MIXED_TOL


def test_lunar_step_overlaps():
    """the grouping and recon of 20 segments, a seventh of the step on one stream, hide behind the Viss for the most part"""
    best = {}
    for serial in (0, 1):
        with Pipeline(config(geometry=0, nside=128, freq_hz=4e6, segs=20, img_n=0, precision=1, serial_stages=serial)) as p:
            p.set_sky(np.ones(p.plan.npix))
            for _ in range(4):
                p.reset_accumulators()
                t = time.perf_counter()
                p.run_all()
                best[serial] = min(best.get(serial, 1e9), time.perf_counter() - t)
    assert best[0] <= 0.92 * best[1], best
