"""One-sky recon of visibilities that overflow, against the CPU FP64 oracle (needs
a GPU): infinities, NaN and finite values in the same places.  The frequency is
so low that a sky of the largest doubles adds up in phase: real parts overflow
while imaginary ones may not."""
import numpy as np
import pytest

from _lockstep import MIXED_TOL, PLAIN_TOL, config, rel_err, run_both

pytestmark = pytest.mark.gpu


def _classes(x):
    return np.where(np.isnan(x), 3, np.where(np.isposinf(x), 2, np.where(np.isneginf(x), 1, 0)))


# (precision, sky): infinite parts; finite parts whose magnitude, or eight times it, overflows; the same in FP32
@pytest.mark.parametrize("mixed,level,kw", [
    (0, 1.7e308, {}), (0, 1.7e308, dict(blockage=0)), (0, 1.7e308, dict(occ_mode=1)), (0, 2.0e307, {}), (0, 1.0e306, {}),
    (1, 5.0e37, {}), (1, 1.0e36, {}),
])
def test_overflow(mixed, level, kw):
    cfg = config(nside=8, n_ant=3, n_epochs=2, segs=1, img_n=21, freq_hz=1.0, precision=mixed, **kw)
    sky = level * np.random.default_rng(1).uniform(0.5, 1.0, 768)
    with np.errstate(all="ignore"):
        (C, W, img, wi), (Co, Wo, imgo, wio) = run_both(cfg, sky)
    assert np.array_equal(W, Wo) and np.array_equal(wi, wio)
    if mixed:  # the oracle's visibilities are FP64: where FP32 held everything, the maps agree
        assert not np.isnan(C).any()
        ok = np.isfinite(C)
        assert ok[W == 0].all() and (level > 1e37 or ok.all())
        assert rel_err(C[ok], Co[ok]) <= MIXED_TOL
        return
    assert np.array_equal(_classes(C), _classes(Co)) and np.array_equal(_classes(img), _classes(imgo))
    fin = np.isfinite(Co)
    if Co[fin].any():
        assert rel_err(C[fin], Co[fin]) <= PLAIN_TOL
