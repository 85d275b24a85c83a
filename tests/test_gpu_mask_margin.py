"""Occlusion masks where a tile's cone finds an antenna's frame all visible by
less than rounding and a point at its far end fails its own test: with a partner
that sees the tile in part, the pair's masks in the one-sky mixed form are the
per-point tests of both, as in the CPU oracle (needs a GPU).

The geometry was found by search: of epoch 5102's antennas, number 3 lies in the
plane of a tile's axis and farthest point, and the altitude puts its horizon
between the cone's bound and that point, 1e-15 apart."""
import numpy as np
import pytest

from _lockstep import MIXED_TOL, config, rel_err
from oracle.oracle import Oracle
from viss_optimize_ws_amd import Pipeline

EPOCH, POINT = 5102, 565606
KW = dict(nside=1, img_n=1024, n_ant=33, n_epochs=EPOCH + 1, segs=EPOCH + 1, orbit_seed=2, freq_hz=1e7, healpix_out=0,
          occ_altitude_km=1022.2351286209323)


def test_bound_with_margin():
    """the geometry does what it says, and the oracle's own bound (bit 0) is no proof that the point is seen"""
    with Oracle(config(**KW)) as o:
        o.gen_segment(EPOCH, 1)
        cls = o.tile_classes(True)[:, POINT // 256].reshape(-1)
        idx, l, m, n = o.img_points()
        x = o.positions()[:, EPOCH]
    a, b = np.triu_indices(33, 1)
    partners = {p for p in (11, 15, 18) if cls[(a == 3) & (b == p)][0] == 0}
    assert partners == {11, 15, 18}  # mixed: partly visible from one of the two at least
    q = 6371.0 / (6371.0 + KW["occ_altitude_km"])
    seen = (np.array([l[POINT], m[POINT], n[POINT]]) @ x) / np.sqrt((x * x).sum(0)) + np.sqrt(1 - q * q)
    assert abs(seen[3]) < 1e-14 and (seen[[11, 15, 18]] > 0).all()


@pytest.mark.gpu
def test_point_behind_a_rounded_bound():
    sky = np.random.default_rng(1).lognormal(0.0, 1.0, 12)
    out = []
    for ctx in (Oracle(config(**KW)), Pipeline(config(precision=1, **KW))):
        with ctx as x:
            x.set_sky(sky)
            x.gen_segment(EPOCH, 1)
            x.viss_half()
            x.conj_fill()
            x.recon_segment()
            out.append(x.finalize())
    (_, _, imgo, wo), (_, _, img, w) = out
    assert np.array_equal(w, wo), (np.argwhere(w != wo)[:4], int((w != wo).sum()))
    assert rel_err(img, imgo) <= MIXED_TOL
