"""The one-launch slice loop adds a detector's sum over the wavefronts of a block
in double, as the tile sums of the passes are added: one bright pixel and faint
ones in the other wavefronts' columns (8 of them each), every value a power of
two, so the sum is known exactly and float32 additions one after the other would
drop each faint one (2^-25 of the bright one, half a unit of rounding).  The
result is the exact sum rounded once."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs

from helpers import random_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nwave", [(64, 64, 1), (96, 64, 130), (64, 128, 130), (128, 128, 130)])
def test_wavefront_sums_in_double(nx, ny, nwave):
    sp = random_setup(nx, ny, nslices=2, nvar=(1, 1), ndetper=1, seed=nx)
    probe = np.zeros((ny, nx), np.complex64)
    faint = np.arange(8, nx, 8)
    probe[ny // 3, faint] = 2.0 ** -13 * (1 + 1j)
    probe[0, 0] = 1
    ones = (np.ones((ny, nx), np.float32), None)
    eng = Engine().setup(configs.Setup(**{**sp.__dict__, "probe": probe, "detectors": [ones]}))
    x = np.zeros(nwave, np.float32)
    eng.stage_scan(x, x, None, np.ones(1, np.float32), np.zeros((nwave, 2), np.int32))
    eng.run_staged(0, nwave)
    eng.sync()
    out = eng.scan_results()
    eng.close()
    want = np.float32(1 + len(faint) * 2.0 ** -25)
    assert want > 1 and (out[:, 0, 0] == want).all(), f"{out[0, 0, 0]:.9f} for {want:.9f}"
