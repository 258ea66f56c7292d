"""Forms of the band-limited and of the split launches that no other test takes.
The real-space readout of one wave in the band-limited row pass, in the small
shape and in the one that columns of 1024 and 2048 points keep: against the
general path (a value of 1e-30 in the propagators' gap), within 1e-6 of the
largest value, as sums differ only in rounding.  And the allocation-free entry
with batches of 40 MiB stored and more, which go in two halves on two streams
once a staged scan has made the second one: against the staged scan, 1e-6
likewise."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs

from helpers import random_setup
from test_zz_no_alloc import _Hip, _noalloc

pytestmark = pytest.mark.gpu
TOL = 1e-6
IMAGE, WAVEREAL = 2, 8


def _close(a, b, what):
    d = np.abs(a - b).max() / np.abs(b).max()
    assert d <= TOL, f"{what}: {d:.2e}"


@pytest.mark.parametrize("nx,ny", [(96, 1024), (1024, 1024), (64, 2048), (2048, 64), (512, 512), (625, 360)])
def test_real_space_readout_of_band_limited_waves(nx, ny):
    sp = random_setup(nx, ny, nslices=4, nvar=(2, 2), ndetper=2, seed=nx + 3 * ny, flags=1 | IMAGE | WAVEREAL)
    pros = []
    for p in sp.propagators:
        p = np.array(p, np.complex64)
        p[:, nx // 2 - 1:nx // 2 + 1] += np.complex64(1e-30)
        p[ny // 2 - 1:ny // 2 + 1, :] += np.complex64(1e-30)
        pros.append(p)
    var, got = configs.variant_sequences(sp, 1, seed=6), []
    for s in (sp, configs.Setup(**{**sp.__dict__, "propagators": pros})):
        eng = Engine().setup(s)
        out = []
        for islc0 in (0, 1):
            eng.wave_offset(0.1, 0.2, 0.0)  # zero in the band's columns from the start
            eng.multislice(var[0], 0.5, False, islc0)
            out += [eng.result(1), eng.result(IMAGE), eng.result(WAVEREAL)]
        out.append(eng.wave_get())
        got.append(out)
        eng.close()
    for k, (a, b) in enumerate(zip(*got)):
        _close(a, b, f"output {k}")


@pytest.mark.parametrize("nx,ny,nwave", [(256, 256, 130), (512, 512, 49), (512, 512, 160), (625, 625, 45),
                                         (640, 720, 62), (1024, 1024, 41)])
def test_allocation_free_entry_in_halves(nx, ny, nwave):
    sp = random_setup(nx, ny, nslices=3, nvar=(2, 2), ndetper=2, seed=nx + 5 * ny)
    rng = np.random.default_rng(nwave)
    dx, dy = rng.uniform(0, 0.4, (2, nwave)).astype(np.float32)
    var, w = configs.variant_sequences(sp, nwave, seed=6), np.ones(1, np.float32)
    eng = Engine().setup(sp)
    eng.set_batch(max(1, (8 << 20) // (8 * nx * ny)))  # one stream, one part
    eng.stage_scan(dx, dy, None, w, var)
    eng.run_staged(0, nwave)
    eng.sync()
    want = eng.scan_results()
    for _ in range(3):
        _close(_noalloc(eng, _Hip(), nwave, 1, dx, dy, w, var), want, "halves")
    eng.close()
