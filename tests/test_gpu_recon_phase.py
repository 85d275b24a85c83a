"""The mixed recon where a segment's rows span no plane: the fitted slopes are
rounding noise of 1e7 and more, phases pass 2^30 turns, and a term has to take
the fraction of the oracle's own FP64 phase before the visibility's argument
comes in (needs a GPU).

Tolerance: a map is a mean of terms |V| cos; the FP32 fraction (2^-25 turns, 2e-7
rad), the FP32 sine and cosine (about 1e-6) and the mixed visibilities (up to
1e-6) leave under 5e-6 of the peak.  Frequencies keep phases below 2^41 turns, to
where the oracle's table index is exact."""
import numpy as np
import pytest

from _lockstep import config, rel_err, run_both

pytestmark = pytest.mark.gpu

TOL = 5e-6


@pytest.mark.parametrize("kw", [
    dict(n_ant=2, n_epochs=1, segs=1, orbit_seed=11),
    dict(n_ant=2, n_epochs=2, segs=2, orbit_seed=5),
    dict(n_ant=2, n_epochs=33, seg_tlen=[16, 1, 16], orbit_seed=10),
    dict(n_ant=2, n_epochs=1, segs=1, orbit_seed=11, recon_mode=1, occ_mode=1),
    dict(n_ant=2, n_epochs=1, segs=1, orbit_seed=11, blockage=0),
], ids=["one", "two", "between", "full_occ1", "blockage0"])
def test_one_row_segments_mixed(kw):
    cfg = config(nside=16, img_n=37, freq_hz=1e6, precision=1, **kw)
    slopes = []
    (C, W, img, wi), (Co, Wo, imgo, wio) = run_both(
        cfg, np.random.default_rng(2).lognormal(0.0, 1.0, 12 * 256),
        lambda g, o, k, d: slopes.append((abs(d["io"]["fa"]) + abs(d["io"]["fb"])) * d["io"]["half"] * d["io"]["du"]))
    assert 2.0 ** 30 < max(slopes) < 2.0 ** 41, slopes
    assert np.array_equal(W, Wo) and np.array_equal(wi, wio)
    assert rel_err(C, Co) <= TOL and rel_err(img, imgo) <= TOL, (rel_err(C, Co), rel_err(img, imgo))
