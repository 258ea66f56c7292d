"""The channels and the exit wave of a wave that is not finite: a grating value
that is no number spreads over the whole plane, also beyond the propagators' band
limit, where the product with the zero propagator is no number either.  Where the
passes leave columns and rows out, the same pixels are not finite as in the
general path (a value of 1e-30 in the propagators' gap), the others agree within
1e-6 of the largest value.  A second run goes on from the exit wave."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs

from helpers import random_setup

pytestmark = pytest.mark.gpu
CHANNELS = (4, 16, 64, 256)  # diffraction, Fourier-space wave, their averages


def _general(sp):
    pros = []
    for p in sp.propagators:
        p = np.array(p, np.complex64)
        p[:, sp.nx // 2 - 1:sp.nx // 2 + 1] += np.complex64(1e-30)
        p[sp.ny // 2 - 1:sp.ny // 2 + 1, :] += np.complex64(1e-30)
        pros.append(p)
    return configs.Setup(**{**sp.__dict__, "propagators": pros})


def _outputs(sp, var, descan):
    eng = Engine().setup(sp)
    eng.set_descan(*descan)
    out = []
    eng.wave_offset(0.1, 0.2, 0.0)
    for again in (False, True):
        eng.multislice(var, 0.5, again)
        out += [eng.result(f) for f in (1, 4, 16) if sp.flags & f]
        out += [eng.avg_result(f)[0] for f in (64, 256) if sp.flags & f]
        out.append(eng.wave_get())
    eng.close()
    return out


@pytest.mark.parametrize("descan", [(0, 0), (5, -3)])
@pytest.mark.parametrize("flags", [1, 1 | sum(CHANNELS)])
@pytest.mark.parametrize("nx,ny", [(64, 64), (64, 96), (96, 128), (256, 256), (512, 512), (625, 360), (96, 1024),
                                   (1024, 1024), (64, 2048)])
def test_channels_of_a_wave_that_is_not_finite(nx, ny, flags, descan):
    sp = random_setup(nx, ny, nslices=3, nvar=(1, 1), ndetper=1, seed=nx + ny, flags=flags)
    gratings = [np.array(g, np.complex64) for g in sp.gratings]
    gratings[1][0, ny // 3, nx // 5] = np.nan  # the second slice's
    var = np.zeros(3, np.int32)
    for g in (sp.gratings, gratings):
        s = configs.Setup(**{**sp.__dict__, "gratings": g})
        a, b = _outputs(s, var, descan), _outputs(_general(s), var, descan)
        for k, (x, y) in enumerate(zip(a, b)):
            fx, fy = np.isfinite(x), np.isfinite(y)
            assert (fx == fy).all(), f"output {k}: {np.sum(fx != fy)} pixels differ in being finite"
            if fx.any():
                d = np.abs(x[fx] - y[fx]).max() / max(np.abs(y[fx]).max(), 1e-30)
                assert d <= 1e-6, f"output {k}: {d:.2e}"
