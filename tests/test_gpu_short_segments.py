"""Whole steps whose consecutive short segments share their launches, against
the same schedule stage by stage, which takes every segment by itself (needs a
GPU).  Weights must be equal; the maps hold the same FP64 terms in another order
of their partial sums (at most 4,096 groups a segment, 2^-53 each: below 1e-12
of the terms' magnitudes, which exceed the maps' peak by less than 100), so
1e-10 of the peak; the mixed form's FP32 block sums are cut elsewhere too and
keep their own bar.  Afterwards the stage calls find the schedule's last segment
as after a step of single segments."""
import numpy as np
import pytest

from _lockstep import MIXED_TOL, config, rel_err
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu

CASES = {
    "four": dict(nside=16, n_ant=8, n_epochs=64, segs=4, img_n=48),
    # lengths on both sides of 1,024 rows: 28 x 36 = 1,008 joins, 28 x 37 = 1,036 does not
    "edge": dict(nside=16, n_ant=8, img_n=40, seg_tlen=[36, 1, 37, 5, 36, 2], n_epochs=117),
    # more short segments than one launch takes, one-row segments among them
    "many": dict(nside=8, n_ant=2, img_n=33, seg_tlen=[1, 3, 2] * 13, n_epochs=78),
    # both halves of the grid, first members with the finite filter, 512-pixel tiles
    "full_occ1": dict(nside=16, n_ant=7, n_epochs=33, segs=5, img_n=45, recon_mode=1, occ_mode=1, tile_pix=512),
    # the antenna-factorized Viss over the run
    "factorized": dict(nside=32, n_ant=16, n_epochs=23, segs=4, img_n=64),
    "mixed": dict(nside=16, n_ant=11, n_epochs=37, segs=5, img_n=61, precision=1),
    # rules and budgets that keep the segments single
    "blockage0": dict(nside=16, n_ant=6, n_epochs=20, segs=4, img_n=32, blockage=0),
    "members": dict(nside=16, n_ant=6, n_epochs=20, segs=4, img_n=32, occ_mode=0),
    "tile_passes": dict(nside=16, n_ant=8, n_epochs=20, segs=4, img_n=32, class_budget_bytes=1),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_step_equals_stages(case):
    kw = CASES[case]
    tol = MIXED_TOL if kw.get("precision") else 1e-10
    with Pipeline(config(**kw)) as a, Pipeline(config(**kw)) as b:
        sky = np.random.default_rng(5).lognormal(0.0, 1.0, a.plan.npix)
        a.set_sky(sky)
        b.set_sky(sky)
        for step in range(2):  # the second on buffers in the other order
            a.reset_accumulators()
            b.reset_accumulators()
            a.run_all()
            for t0, tl in b.schedule():
                b.gen_segment(t0, tl)
                b.viss_half()
                b.conj_fill()
                ib = b.recon_segment()
            Ca, Wa, Ia, WIa = a.finalize()
            Cb, Wb, Ib, WIb = b.finalize()
            assert np.array_equal(Wa, Wb) and np.array_equal(WIa, WIb), (case, step)
            assert rel_err(Ca, Cb) <= tol and rel_err(Ia, Ib) <= tol, (case, step, rel_err(Ca, Cb), rel_err(Ia, Ib))
        ia = a.recon_segment()  # of the last segment
        assert (ia["t0"], ia["tlen"], ia["nuniq"], ia["nkeys"]) == (ib["t0"], ib["tlen"], ib["nuniq"], ib["nkeys"])
