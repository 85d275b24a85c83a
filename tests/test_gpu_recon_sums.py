"""Rounding of the plain recon's sums where one range holds a whole segment's
groups: 8.5 million points in one pass, 77,658 groups (needs a GPU).

Reference: the same sum over the context's own group visibilities in extended
precision, at 100 points.  What the kernel's arithmetic leaves, in units of the
rms visibility: phases of up to 512 turns, rounded at four places (1.6e-13 rad a
term, 4.4e-11 over 77,658 terms), the cosine's 1.9e-13 at most (3.6e-11), and
signed partial sums of about a thousand (1e-11): 6e-11, a few times that at
most.  Sums left to cancel at the end of the range reach 77,658, and their
roundings 1.1e-9.  The bound lies between."""
import numpy as np
import pytest

from _lockstep import config
from viss_optimize_ws_amd import Pipeline

pytestmark = pytest.mark.gpu


def test_long_range_of_groups():
    n = 833
    cfg = config(nside=4, n_ant=16, n_epochs=n, segs=1, img_n=3300, freq_hz=4e3, blockage=0, healpix_out=0,
                 class_budget_bytes=7 << 30)
    with Pipeline(cfg) as p:
        p.set_sky(np.random.default_rng(3).lognormal(0.0, 1.0, p.plan.npix))
        p.gen_segment(0, n)
        p.viss_half()
        half, _ = p.conj_fill()
        p.recon_segment()
        info, keys, off, order, _ = p.groups()
        _, _, G, _, total = p.accumulators()
        _, l, m, nn = p.img_points()
    assert total == info["nuniq"] > 60000
    V = np.add.reduceat(half[order], off[:-1]) / np.diff(off)
    live = keys > 0
    key, V = keys[live] - 1, V[live]
    L = np.longdouble
    u = ((key // info["res"] - info["half"]) * info["du"]).astype(L)
    v = ((key % info["res"] - info["half"]) * info["du"]).astype(L)
    amp, arg = np.abs(V).astype(L), np.angle(V).astype(L)
    err = []
    for i in np.random.default_rng(4).choice(l.size, 100, replace=False):
        x = u * (L(l[i]) + L(info["fa"]) * L(nn[i])) + v * (L(m[i]) + L(info["fb"]) * L(nn[i]))
        x -= np.rint(x)
        err.append(float(G[i] - np.sum(amp * np.cos(2 * L("3.14159265358979323846264338328") * x + arg))))
    rms = np.sqrt(np.mean(np.square(err))) / np.sqrt(np.mean(np.abs(V) ** 2))
    print("rms error", rms)
    assert rms <= 4e-10, rms
