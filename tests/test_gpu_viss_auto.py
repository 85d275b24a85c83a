"""The plain form's automatic choice between the per-row and the
antenna-factorized Viss, against the CPU FP64 oracle, and where it must not
take the factorized one (needs a GPU)."""
import numpy as np
import pytest

from _lockstep import PLAIN_TOL, config, rel_err
from oracle.oracle import Oracle
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu


def _viss(cfg, sky):
    with Pipeline(cfg) as g:
        g.set_sky(sky)
        out = []
        for t0, tl in g.schedule():
            g.gen_segment(t0, tl)
            out.append(g.viss_half())
        return np.concatenate(out)


# the ends of the ranges that take it and their neighbours that do not; ragged epochs, both tile sizes, tile passes
@pytest.mark.parametrize("n_ant,tp,budget", [(12, 256, 0), (13, 256, 0), (16, 512, 0), (17, 256, 0), (21, 256, 0),
                                             (22, 512, 0), (32, 256, 0), (32, 256, 40000), (33, 256, 0)])
def test_automatic_form_matches_the_oracle(n_ant, tp, budget):
    cfg = config(nside=32, n_ant=n_ant, n_epochs=7, segs=2, freq_hz=1e7, img_n=0, tile_pix=tp, class_budget_bytes=budget)
    sky = np.random.default_rng(n_ant).lognormal(0.0, 1.0, 12 * 32 * 32)
    v = _viss(cfg, sky)
    with Oracle(cfg) as o:
        o.set_sky(sky)
        ref = []
        for t0, tl in o.schedule():
            o.gen_segment(t0, tl)
            ref.append(o.viss_half())
    assert rel_err(v, np.concatenate(ref)) <= PLAIN_TOL


def test_automatic_form_keeps_rows_for_long_baselines_and_nan():
    """100 MHz (4.7e6 turns) and a sky with a NaN pixel give the row form's bits"""
    kw = dict(nside=16, n_ant=16, n_epochs=5, segs=1, img_n=0)
    sky = np.random.default_rng(1).lognormal(0.0, 1.0, 12 * 256)
    long = config(freq_hz=1e8, **kw), config(freq_hz=1e8, viss_form=1, **kw)
    assert np.array_equal(_viss(long[0], sky), _viss(long[1], sky))
    bad = sky.copy()
    bad[17] = np.nan
    short = config(freq_hz=1e7, **kw), config(freq_hz=1e7, viss_form=1, **kw)
    a, b = _viss(short[0], bad), _viss(short[1], bad)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and 0 < np.isnan(a).sum() < a.size
    assert np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])
