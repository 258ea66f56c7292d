"""Waves that are not finite: a readout sum takes every pixel of its plane, so
one value that is infinite or no number (or whose square overflows) makes every
sum of the plane not finite (0 * inf), also that of a detector without a weight
in its column or anywhere, in each of the readout's kernels and with the
band-limited forms as with the general one."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs

from helpers import random_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.nan, np.inf, 1e30])
@pytest.mark.parametrize("nx,ny", [(64, 64), (160, 96), (256, 256), (480, 625), (96, 1024)])
def test_sums_are_not_finite(nx, ny, value):
    sp = random_setup(nx, ny, nslices=2, nvar=(1, 1), ndetper=1, seed=nx)
    none = (np.zeros((ny, nx), np.float32), None)
    sp = configs.Setup(**{**sp.__dict__, "detectors": [*sp.detectors, none]})
    col = 1 + np.flatnonzero(np.abs(np.asarray(sp.detectors[0][0])).sum(0)[1:nx // 4] == 0)[0]
    probe = np.array(sp.probe, np.complex64)
    probe[ny // 5, col] = value  # inside the band; detector 0 has no weight in this column
    eng = Engine().setup(configs.Setup(**{**sp.__dict__, "probe": probe}))
    x = np.zeros(200, np.float32)
    eng.stage_scan(x, x, None, np.ones(1, np.float32), np.zeros((200, 2), np.int32))
    for n in (2, 200):  # the small launch shapes, and those of the length
        eng.run_staged(0, n)
        eng.sync()
        out = eng.scan_results()[:n]
        assert not np.isfinite(out).any(), f"{n} waves: {out[0]}"
    eng.wave_set(probe)
    eng.multislice(np.zeros(2, np.int32), 1.0)
    assert not np.isfinite(eng.result(1)).any()
    eng.close()


@pytest.mark.parametrize("nx,ny", [(64, 64), (256, 256), (96, 1024)])
def test_phase_plate_is_not_finite(nx, ny):
    """The constant phase plate multiplies every column of the incident wave,
    also those where the probe and the propagators are zero."""
    sp = random_setup(nx, ny, nslices=2, nvar=(1, 1), ndetper=1, seed=nx)
    plate = np.zeros((ny, nx), np.float32)
    plate[ny // 3, nx // 2] = np.nan
    x = np.zeros(200, np.float32)
    eng = Engine().setup(sp)
    eng.stage_scan(x, x, None, np.ones(1, np.float32), np.zeros((200, 2), np.int32))
    for p in (None, plate, None):
        eng._c("jms_hip_set_phaseplate", None if p is None else p.ctypes.data)
        for n in (2, 200):
            eng.run_staged(0, n)
            eng.sync()
            out = eng.scan_results()[:n]
            assert np.isfinite(out).all() if p is None else not np.isfinite(out).any(), f"{n} waves"
    eng._c("jms_hip_set_phaseplate", plate.ctypes.data)
    eng.wave_offset(0.0, 0.0)
    eng._c("jms_hip_set_phaseplate", None)  # the wave has it already
    eng.multislice(np.zeros(2, np.int32), 1.0)
    assert not np.isfinite(eng.result(1)).any()
    eng.close()
