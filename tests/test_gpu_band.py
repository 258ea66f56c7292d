"""Band-limited waves: where every propagator of a run vanishes, the passes
leave the columns (and the transforms the rows) out.  The same set-up with a
value of 1e-30 at the centre of the propagators takes the general path, which
keeps every column; both compute the same sums on the columns that count, so
results agree to float32 rounding (the instantiations may contract products
differently; 1e-6 of the largest value, 20 times float32's unit rounding)."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, Group, configs

from helpers import random_setup

pytestmark = pytest.mark.gpu
TOL = 1e-6


def _general(sp):
    """The same set-up without a zero gap in its propagators."""
    pros = []
    for p in sp.propagators:
        p = np.array(p, np.complex64)
        p[:, sp.nx // 2 - 1:sp.nx // 2 + 1] += np.complex64(1e-30)
        p[sp.ny // 2 - 1:sp.ny // 2 + 1, :] += np.complex64(1e-30)
        pros.append(p)
    return configs.Setup(**{**sp.__dict__, "propagators": pros})


def _close(a, b, what):
    d = np.abs(a - b).max() / np.abs(b).max()
    assert d <= TOL, f"{what}: {d:.2e}"


def _scan(sp, var, dx, dy, graph=False, islc0=0, descan=(0, 0)):
    eng = Engine().setup(sp)
    eng.set_graph(graph)
    eng.set_descan(*descan)
    eng.stage_scan(dx, dy, None, np.ones(1, np.float32), var)
    out = []
    for _ in range(2 if graph else 1):
        eng.run_staged(0, len(dx), islc0)
        eng.sync()
        out.append(eng.scan_results())
    eng.close()
    return out[-1]


SIZES = [(16, 16), (64, 64), (96, 128), (128, 96), (192, 160), (256, 256), (320, 360), (360, 320), (384, 384),
         (480, 480), (512, 512), (625, 625), (640, 640), (720, 720), (768, 768), (1024, 360), (360, 1024),
         (2048, 96), (64, 2048), (625, 1024)]


@pytest.mark.parametrize("nx,ny", SIZES)
def test_band_equals_general_path(nx, ny):
    sp = random_setup(nx, ny, nslices=5, nvar=(2, 2), ndetper=2, seed=nx + 3 * ny, flags=1 | 4 | 16)
    ref = _general(sp)
    var = configs.variant_sequences(sp, 3, seed=6)
    dx, dy = np.array([0.0, 0.11, 0.3], np.float32), np.array([0.2, 0.0, 0.07], np.float32)
    _close(_scan(sp, var, dx, dy), _scan(ref, var, dx, dy), "staged scan")
    got = []
    for s in (sp, ref):  # one wave: readouts, channels and the exit wave with its cleared columns
        eng = Engine().setup(s)
        eng.wave_set(np.random.default_rng(3).standard_normal((ny, nx, 2)).astype(np.float32).view(np.complex64)[..., 0])
        eng.multislice(var[0], 0.5)
        got.append((eng.result(1), eng.result(4), eng.result(16), eng.wave_get()))
        eng.close()
    for a, b, what in zip(*got, ("sums", "diffraction", "Fourier-space wave", "exit wave")):
        _close(a, b, what)


def test_band_options():
    """Graph replay, a start plane, de-scan, a probe with content in the gap,
    a second propagator with a wider band, and set-ups that change the band
    of an engine between runs."""
    nx = ny = 256
    sp = random_setup(nx, ny, nslices=6, nvar=(2, 2), ndetper=3, seed=5)
    var = configs.variant_sequences(sp, 2, seed=6)
    dx, dy = np.array([0.0, 0.11], np.float32), np.array([0.2, 0.0], np.float32)
    ref = _general(sp)
    for kw in (dict(graph=True), dict(islc0=3), dict(islc0=6), dict(descan=(5, -9))):
        _close(_scan(sp, var, dx, dy, **kw), _scan(ref, var, dx, dy, **kw), str(kw))
    rng = np.random.default_rng(1)
    full = (rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))).astype(np.complex64) / nx
    wide = configs.Setup(**{**sp.__dict__, "probe": full})
    _close(_scan(wide, var, dx, dy), _scan(_general(wide), var, dx, dy), "probe with content in the gap")
    p2 = np.array(sp.propagators[0], np.complex64)
    p2[:, 100:110] = p2[:, :10]  # live columns inside the first propagator's gap
    two = configs.Setup(**{**sp.__dict__, "propagators": [sp.propagators[0], p2], "proidx": [0, 1]})
    _close(_scan(two, var, dx, dy), _scan(_general(two), var, dx, dy), "two propagators")
    a, b = Engine().setup(sp), Engine().setup(_general(two))  # b holds the general path of `two`
    for eng in (a, b):
        eng.set_graph(True)
    for s in (sp, two, wide):
        g = _general(s)
        a.setup(s), b.setup(g)
        for eng in (a, b):
            eng.stage_scan(dx, dy, None, np.ones(1, np.float32), var)
            eng.run_staged(0, 2)
            eng.sync()
        _close(a.scan_results(), b.scan_results(), "set up again")
    a.close(), b.close()


def test_band_of_a_group():
    """Members whose bands differ (one with a wider propagator, one whose
    probe has content in the gap) share the columns that all of them leave out."""
    rng = np.random.default_rng(2)
    sps = [random_setup(256, 256, nslices=k, nvar=(1, 1), ndetper=2, seed=k) for k in (5, 3, 4)]
    p2 = np.array(sps[1].propagators[0], np.complex64)
    p2[:, 100:110] = p2[:, :10]
    wide = configs.Setup(**{**sps[1].__dict__, "propagators": [p2, sps[1].propagators[1]]})
    full = (rng.standard_normal((256, 256)) + 1j * rng.standard_normal((256, 256))).astype(np.complex64) / 256
    odd = configs.Setup(**{**sps[2].__dict__, "probe": full})
    dx, dy = np.array([0.0, 0.1], np.float32), np.array([0.2, 0.3], np.float32)
    for members in ((sps[0], sps[1], sps[2]), (sps[0], wide, sps[2]), (sps[0], wide, odd)):
        engines = []
        for sp in members:
            eng = Engine().setup(sp)
            eng.stage_scan(dx, dy, None, np.ones(1, np.float32), np.zeros((2, len(sp.objslc)), np.int32))
            engines.append(eng)
        grp = Group(engines)
        grp.run()
        grp.sync()
        for sp, eng in zip(members, engines):
            ref = _scan(_general(sp), np.zeros((2, len(sp.objslc)), np.int32), dx, dy)
            _close(eng.scan_results(), ref, "member")
        grp.close()
        for eng in engines:
            eng.close()


@pytest.mark.parametrize("nx,ny", [(16, 32), (32, 16), (64, 64), (96, 128), (128, 96), (256, 256), (320, 360),
                                   (384, 480), (512, 512), (625, 625), (640, 640), (720, 720), (768, 64), (64, 768)])
def test_small_launches_equal_large_ones(nx, ny):
    """A batch that leaves CUs without a block takes the small launch shapes
    (natural layout, other column tiles), a larger one the shapes of the line
    length (panels where it has them), with and without a band."""
    sp = random_setup(nx, ny, nslices=4, nvar=(2, 2), ndetper=2, seed=nx + ny)
    few, many = 3, 256 // max(1, nx // 16) + 3  # column tiles are at most 16 wide
    var = np.resize(configs.variant_sequences(sp, few, seed=6), (many, 4))
    x, y = np.array([0.0, 0.11, 0.3], np.float32), np.array([0.2, 0.0, 0.07], np.float32)
    for s in (sp, _general(sp)):
        small = _scan(s, var[:few], x, y)
        large = _scan(s, var, np.resize(x, many), np.resize(y, many))
        _close(large, small[np.resize(np.arange(few), many)], "large against small launches")
