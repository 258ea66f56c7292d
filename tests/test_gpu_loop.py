"""The slice loop of small waves in one launch: batches that take it against
the row and column passes (the single-wave path with a diffraction channel
keeps those), on every grid the kernel exists for, with and without a band.
Both compute the same transforms; sums are taken in another order, so every
intensity agrees within 1e-6 of the largest (20 times float32's unit
rounding).  One case is also checked against the oracle."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs
from oracle import oracle as O

from helpers import assert_dets, random_setup

pytestmark = pytest.mark.gpu
TOL = 1e-6
X, Y = np.array([0.0, 0.11, 0.3], np.float32), np.array([0.2, 0.0, 0.07], np.float32)


def _general(sp):
    pros = []
    for p in sp.propagators:
        p = np.array(p, np.complex64)
        p[:, sp.nx // 2] += np.complex64(1e-30)
        pros.append(p)
    return configs.Setup(**{**sp.__dict__, "propagators": pros})


def _passes(sp, var, islc0=0, descan=(0, 0), plate=None):
    eng = Engine().setup(configs.Setup(**{**sp.__dict__, "flags": 1 | 4}))
    eng.set_descan(*descan)
    if plate is not None:
        eng._c("jms_hip_set_phaseplate", plate.ctypes.data)
    out = []
    for k in range(3):
        eng.wave_offset(float(X[k]), float(Y[k]), 0.0)
        eng.multislice(var[k], 1.0, False, islc0)
        out.append(eng.result(1))
    eng.close()
    return np.stack(out)


def _staged(sp, var, nw, islc0=0, descan=(0, 0), plate=None, graph=False):
    eng = Engine().setup(sp)
    eng.set_descan(*descan)
    eng.set_graph(graph)
    if plate is not None:
        eng._c("jms_hip_set_phaseplate", plate.ctypes.data)
    eng.stage_scan(np.resize(X, nw), np.resize(Y, nw), None, np.ones(1, np.float32), np.resize(var, (nw, var.shape[1])))
    for _ in range(3 if graph else 1):
        eng.run_staged(0, nw, islc0)
        eng.sync()
        out = eng.scan_results()
    eng.close()
    return out


def _close(a, b, what):
    d = np.abs(a - b).max() / np.abs(b).max()
    assert d <= TOL, f"{what}: {d:.2e}"


@pytest.mark.parametrize("nx", [64, 96, 128])
@pytest.mark.parametrize("ny", [64, 96, 128])
def test_loop_equals_passes(nx, ny):
    sp = random_setup(nx, ny, nslices=5, nvar=(2, 2), ndetper=2, seed=nx + 3 * ny)
    var = configs.variant_sequences(sp, 3, seed=6)
    for s in (sp, _general(sp)):
        ref = _passes(s, var)
        for nw in (3, 130):
            _close(_staged(s, var, nw), ref[np.resize(np.arange(3), nw)], f"{nw} waves")


def test_loop_options():
    nx, ny = 64, 96
    sp = random_setup(nx, ny, nslices=6, nvar=(2, 2), ndetper=3, seed=5)
    var = configs.variant_sequences(sp, 3, seed=6)
    plate = np.random.default_rng(3).uniform(-1, 1, (ny, nx)).astype(np.float32)
    for kw in (dict(islc0=3), dict(islc0=6), dict(descan=(5, -9)), dict(plate=plate)):
        _close(_staged(sp, var, 130, **kw), _passes(sp, var, **kw)[np.resize(np.arange(3), 130)], str(kw.keys()))
    _close(_staged(sp, var, 130, graph=True), _passes(sp, var)[np.resize(np.arange(3), 130)], "graph")
    rng = np.random.default_rng(1)
    full = (rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))).astype(np.complex64) / nx
    wide = configs.Setup(**{**sp.__dict__, "probe": full})
    _close(_staged(wide, var, 130), _passes(wide, var)[np.resize(np.arange(3), 130)], "probe with content in the gap")
    w = np.array([0.3, 0.7], np.float32)
    eng = Engine().setup(sp)
    v2 = configs.variant_sequences(sp, 130, seed=9)
    x, y = np.linspace(0, 0.4, 65).astype(np.float32), np.linspace(0, 0.3, 65).astype(np.float32)
    eng.stage_scan(x, y, None, w, v2)
    eng.run_staged(0, 65)
    eng.sync()
    ref = O.stem_scan(sp, x, y, w, v2, prec=32, nthreads=4)
    assert_dets(eng.scan_results(), ref, 1e-4, "two passes per position")
    eng.close()


def test_single_wave_keeps_the_exit_wave():
    sp = random_setup(64, 64, nslices=5, nvar=(2, 2), seed=8)
    var = configs.variant_sequences(sp, 1, seed=6)
    got = []
    for flags in (1, 1 | 4):  # one launch; the passes
        for s in (sp, _general(sp)):
            eng = Engine().setup(configs.Setup(**{**s.__dict__, "flags": flags}))
            eng.wave_offset(0.1, 0.2, 0.0)
            eng.multislice(var[0], 0.5)
            eng.multislice(var[0], 0.5, accumulate=True)  # on from the exit wave
            got.append((eng.result(1), eng.wave_get()))
            eng.close()
    for g in got[1:]:
        _close(g[0], got[0][0], "sums")
        _close(g[1], got[0][1], "exit wave")
