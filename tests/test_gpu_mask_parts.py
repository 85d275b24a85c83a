"""The masks of the one-sky recon where several workgroups share a tile (few
tiles, more than 512 antenna frames), against the CPU FP64 oracle and the stage
calls, and that such recons take no longer than their work (needs a GPU)."""
import numpy as np
import pytest

from _lockstep import MIXED_TOL, config, rel_err, run_both
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu


# frames: 512 (one workgroup), 513, 1,024, 1,025 (two, two, three), 32,768 and 32,770 (cone bits in LDS, from the table)
@pytest.mark.parametrize("kw", [dict(n_ant=2, n_epochs=256), dict(n_ant=3, n_epochs=171), dict(n_ant=4, n_epochs=256),
                                dict(n_ant=5, n_epochs=205), dict(n_ant=2, n_epochs=16384, dt_s=1.0),
                                dict(n_ant=2, n_epochs=16385, dt_s=1.0), dict(n_ant=7, n_epochs=200, tile_pix=512),
                                dict(n_ant=6, n_epochs=190, recon_mode=1, occ_mode=1, class_budget_bytes=300000)])
def test_shared_tiles(kw):
    cfg = config(nside=4, segs=1, img_n=21, freq_hz=1e7, precision=1, **kw)
    sky = np.random.default_rng(6).lognormal(0.0, 1.0, 12 * 16)
    (C, W, img, wi), (Co, Wo, imgo, wio) = run_both(cfg, sky)
    assert np.array_equal(W, Wo) and np.array_equal(wi, wio)
    assert rel_err(C, Co) <= MIXED_TOL and rel_err(img, imgo) <= MIXED_TOL


def test_plain_tables_shared():
    """plain, groups of a tile shared (cone bits from the table): weights and maps"""
    cfg = config(nside=2, n_ant=2, n_epochs=16500, segs=1, img_n=9, freq_hz=1e7, dt_s=1.0)
    (C, W, img, wi), (Co, Wo, imgo, wio) = run_both(cfg, np.random.default_rng(7).lognormal(0.0, 1.0, 48))
    assert np.array_equal(W, Wo) and np.array_equal(wi, wio)
    assert rel_err(C, Co) <= 1e-9 and rel_err(img, imgo) <= 1e-9


def test_shared_tiles_of_merged_segments():
    """a step whose short segments share their launches: frames and groups of all of them"""
    kw = dict(nside=8, n_ant=3, img_n=33, seg_tlen=[300, 1, 298, 300, 5, 77], n_epochs=981, precision=1)
    with Pipeline(config(**kw)) as a, Pipeline(config(**kw)) as b:
        sky = np.random.default_rng(8).lognormal(0.0, 1.0, a.plan.npix)
        a.set_sky(sky)
        b.set_sky(sky)
        a.run_all()
        for t0, tl in b.schedule():
            b.gen_segment(t0, tl)
            b.viss_half()
            b.conj_fill()
            b.recon_segment()
        (Ca, Wa, Ia, WIa), (Cb, Wb, Ib, WIb) = a.finalize(), b.finalize()
    assert np.array_equal(Wa, Wb) and np.array_equal(WIa, WIb)
    assert rel_err(Ca, Cb) <= MIXED_TOL and rel_err(Ia, Ib) <= MIXED_TOL


def test_mixed_recon_keeps_up_with_plain():
    """3 tiles and 400,000 frames: the mixed terms cost less than the plain ones, and the frames' occlusion tests about as
    much as the plain form's; with one workgroup a tile the mixed recon took eight times as long as the plain one"""
    best = {}
    for prec in (0, 1):
        with Pipeline(config(nside=8, n_ant=2, n_epochs=200000, segs=1, img_n=0, dt_s=1.0, precision=prec)) as p:
            p.set_sky(np.ones(p.plan.npix))
            p.gen_segment(0, 200000)
            p.viss_half()
            p.conj_fill()
            for _ in range(5):
                t = p.timings()["recon_ms"]
                p.recon_segment()
                best[prec] = min(best.get(prec, 1e9), p.timings()["recon_ms"] - t)
    assert best[1] <= 3.0 * best[0], best
