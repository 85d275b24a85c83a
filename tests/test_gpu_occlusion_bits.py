"""The mixed recon's occlusion bits per antenna frame (queued 64 frames a wave,
cone bits in LDS up to 32,768 frames, 64 points a word) and the one-workgroup
grouping (1,024 rows) at their edges, against the CPU FP64 oracle (needs a GPU).
Weights, keys and groups bit-exact, maps to the mixed bar."""
import numpy as np
import pytest

from _lockstep import MIXED_TOL, config, rel_err, run_both
from oracle.oracle import Oracle
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "kw",
    [dict(n_ant=3, n_epochs=21), dict(n_ant=2, n_epochs=32), dict(n_ant=5, n_epochs=13), dict(n_ant=13, n_epochs=67),
     dict(n_ant=8, n_epochs=40, tile_pix=512), dict(n_ant=9, n_epochs=30, class_budget_bytes=1),
     dict(n_ant=2, n_epochs=16500, nside=2, img_n=9, dt_s=1.0), dict(n_ant=7, n_epochs=25, recon_mode=1, occ_mode=1)],
    ids=["63_frames", "64_frames", "65_frames", "871_frames", "tp512", "tile_passes", "33000_frames", "full_occ1"],
)
def test_mixed_masks(kw):
    base = dict(nside=8, segs=1, img_n=27, freq_hz=1e7, precision=1)
    base.update(kw)
    cfg = config(**base)
    (C, W, img, wi), (Co, Wo, imgo, wio) = run_both(cfg, np.random.default_rng(3).lognormal(0.0, 1.0, 12 * base["nside"] ** 2))
    assert np.array_equal(W, Wo) and np.array_equal(wi, wio)
    assert rel_err(C, Co) <= MIXED_TOL and rel_err(img, imgo) <= MIXED_TOL


@pytest.mark.parametrize("rows,full", [(1, 0), (1, 1), (511, 1), (512, 1), (513, 1), (1023, 0), (1024, 0), (1025, 0)])
def test_one_workgroup_grouping(rows, full):
    """1 MHz and one-second epochs put many rows in a cell: equal keys keep their order"""
    cfg = config(nside=4, n_ant=2, n_epochs=rows, segs=1, img_n=0, freq_hz=1e6, dt_s=1.0, recon_mode=full, occ_mode=1)
    with Pipeline(cfg) as g, Oracle(cfg) as o:
        for x in (g, o):
            x.set_sky(np.ones(12 * 16))
            x.gen_segment(0, rows)
            x.viss_half()
            x.conj_fill()
            x.recon_segment()
        a, b = g.groups(), o.groups()
    for k in ("fa", "fb", "denom", "du", "res", "half", "nuniq", "nkeys"):
        assert a[0][k] == b[0][k], k
    for x, y in zip(a[1:], b[1:]):
        assert np.array_equal(x, y)
