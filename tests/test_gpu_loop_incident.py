"""The incident plane's readout of the one-launch slice loop.  The incident
wave has met no propagator, so it may hold intensity in the rows where every
propagator vanishes (a probe tilted by half the grid, an aperture shifted in y)
while the columns there are zero and the loop leaves them out.  Compared with
the row and column passes (a diffraction channel keeps those) within 1e-6 of
the largest value, 20 times float32's unit rounding: the sums are taken in
another order."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs

from helpers import random_setup

pytestmark = pytest.mark.gpu
TOL = 1e-6


def _close(a, b, what):
    assert np.abs(b[..., 0, :]).max() > 0.1  # the incident plane carries the intensity
    d = np.abs(a - b).max() / np.abs(b).max()
    assert d <= TOL, f"{what}: {d:.2e}"


def _setup(nx, ny):
    """Plane 0 read out, with a detector over the whole plane in the place of
    the second one."""
    sp = random_setup(nx, ny, nslices=4, nvar=(2, 2), ndetper=1, seed=nx + 3 * ny)
    dets = [sp.detectors[0], (np.ones((ny, nx), np.float32), None), sp.detectors[2]]
    return configs.Setup(**{**sp.__dict__, "detectors": dets})


def _single(sp, var, wave, islc0=0):
    out = []
    for flags in (1, 1 | 4):  # one launch; the passes
        eng = Engine().setup(configs.Setup(**{**sp.__dict__, "flags": flags}))
        wave(eng)
        eng.multislice(var, 1.0, False, islc0)
        out.append(eng.result(1))
        eng.close()
    return out


@pytest.mark.parametrize("nx,ny", [(64, 64), (64, 96), (96, 64)])
def test_incident_rows(nx, ny):
    sp = _setup(nx, ny)
    var = configs.variant_sequences(sp, 130, seed=6)
    rng = np.random.default_rng(nx)
    band = np.abs(np.arange(nx) - nx // 2) > nx // 4  # columns outside the gap, every row
    wide = (rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))) * band
    wide = (wide / np.linalg.norm(wide)).astype(np.complex64)
    if nx * ny <= 64 * 64:  # single waves take the loop
        a, b = _single(sp, var[0], lambda e: e.wave_offset(0.1, 0.2, 0.0, 0, ny // 2))
        _close(a, b, "beam tilt by half the rows")
        a, b = _single(sp, var[0], lambda e: e.wave_set(wide))
        _close(a, b, "wave over all rows")
    x, y = rng.uniform(0, 0.3, (2, 130)).astype(np.float32)
    for probe in (wide, np.roll(np.asarray(sp.probe), ny // 2, 0)):
        s = configs.Setup(**{**sp.__dict__, "probe": probe})
        loop = Engine().setup(s)
        loop.stage_scan(x, y, None, np.ones(1, np.float32), var)
        passes = Engine().setup(configs.Setup(**{**s.__dict__, "flags": 1 | 4}))
        for islc0 in (0, 2):
            loop.run_staged(0, 130, islc0)
            loop.sync()
            got, ref = loop.scan_results()[:3, islc0:], []
            for k in range(3):
                passes.wave_offset(float(x[k]), float(y[k]), 0.0)
                passes.multislice(var[k], 1.0, False, islc0)
                ref.append(passes.result(1))
            _close(got, np.stack(ref)[:, islc0:], f"staged scan from plane {islc0}")
        loop.close(), passes.close()
