"""Readouts leave out the detectors without a weight in a column: the sums
equal the diffraction channel times the weights, for detectors that are empty,
hold one pixel, end inside a column tile or cover everything, masked or not,
with a de-scan, and after a detector was replaced.  Sums of up to 2.6e5 float32
terms in partial sums of a few hundred: 1e-5 of the largest sum."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs
from jmultislicelib_amd._lib import ptr

from helpers import random_setup

pytestmark = pytest.mark.gpu


def _mask(d, i):
    return np.flatnonzero(d).astype(np.int32) if i == 2 else None


@pytest.mark.parametrize("nx,ny", [(16, 32), (48, 64), (128, 128), (360, 320), (625, 48), (512, 512), (64, 1024)])
@pytest.mark.parametrize("descan", [(0, 0), (7, -5)])
def test_sums_equal_weighted_diffraction(nx, ny, descan):
    sp = random_setup(nx, ny, nslices=2, nvar=(1, 1), ndetper=1, seed=nx + ny, flags=1 | 4)
    rng = np.random.default_rng(nx)
    one, edge = np.zeros((2, ny, nx), np.float32)
    one[ny - 1, 1] = 2.0
    edge[:, 3:9] = rng.uniform(0.5, 1, (ny, 6))
    dets = [np.zeros((ny, nx), np.float32), one, edge, rng.uniform(0, 1, (ny, nx)).astype(np.float32)]
    sp = configs.Setup(**{**sp.__dict__, "detectors": [(d, _mask(d, i)) for i, d in enumerate(dets)]})
    eng = Engine().setup(sp)
    eng.set_descan(*descan)
    wave = rng.standard_normal((ny, nx, 2)).astype(np.float32).view(np.complex64)[..., 0] / nx
    for swap in (False, True):
        if swap:  # the empty detector gets weights, the full one loses them
            dets[0], dets[3] = dets[3], dets[0]
            for d in (0, 3):
                eng._c("jms_hip_upload_detector", d, ptr(dets[d]), 0, None)
        eng.wave_set(wave)
        eng.multislice(np.zeros(2, np.int32))
        sums, dif = eng.result(1), eng.result(4).astype(np.float64)
        want = np.array([[(p * d).sum() for d in dets] for p in dif])
        assert np.abs(sums - want).max() <= 1e-5 * np.abs(want).max()
        assert (sums[:, 3 if swap else 0] == 0).all()
    eng.close()
