"""Waves in panels whose last one is partly filled (a row length that is no
multiple of 16): staged and grouped batches keep whole panels in their own
buffers, the allocation-free entry works in the caller's, one grid a wave, and
must leave what lies behind it alone.  All compute the same sums (1e-6 of the
largest value: instantiations may contract products differently)."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, Group, configs

from helpers import random_setup
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu
TOL = 1e-6


@pytest.mark.parametrize("nx,ny", [(625, 625), (625, 640), (640, 625), (625, 48)])
def test_partly_filled_panels(nx, ny):
    sp = random_setup(nx, ny, nslices=3, nvar=(2, 2), ndetper=2, seed=nx + ny)
    nwave = 131 if ny < 100 else 5  # more than a small launch (128 column tiles)
    rng = np.random.default_rng(ny)
    dx, dy = rng.uniform(0, 0.4, (2, nwave)).astype(np.float32)
    var = configs.variant_sequences(sp, nwave, seed=2)
    w = np.ones(1, np.float32)
    engines = [Engine().setup(sp) for _ in range(2)]
    for eng in engines:
        eng.stage_scan(dx, dy, None, w, var)
    engines[0].run_staged(0, nwave)
    engines[0].sync()
    staged = engines[0].scan_results()
    grp = Group(engines)
    grp.run()
    grp.sync()
    got = {"group": engines[0].scan_results(), "group's second": engines[1].scan_results()}
    grp.close()
    ppar = np.zeros((nwave, 4), np.float32)
    ppar[:, 0], ppar[:, 1] = dx, dy
    hip = _Hip()
    nw = 2 * nx * ny * nwave
    waves = hip.put(np.full(nw + 64 * ny, 7.0, np.float32))
    res = hip.put(np.zeros(staged.size, np.float32))
    eng = engines[1]
    rc = eng.L.jms_hip_run_batch_noalloc(eng.h, 0, nwave, waves, hip.put(ppar), hip.put(np.asarray(var, np.int32)),
                                         nwave, 1, hip.put(w), res)
    assert rc == 0, eng.L.jms_hip_last_error(eng.h)
    eng.sync()
    got["caller's buffers"] = hip.get(res, staged.shape, np.float32)
    behind = hip.get(waves, (nw + 64 * ny,), np.float32)[nw:]
    hip.free()
    assert (behind == 7.0).all(), "written behind the caller's waves"
    for eng in engines:
        eng.close()
    for what, r in got.items():
        d = np.abs(r - staged).max() / np.abs(staged).max()
        assert d <= TOL, f"{what}: {d:.2e}"
