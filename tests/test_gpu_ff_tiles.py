"""Structure-factor sums of the form-factor gratings at the edges of their
tiles (32 x 32 or, for many, 64 x 64 pixels; 32 atoms at a time): grids that
end inside a tile, atom counts around the chunk, empty sets and missing types,
against the float64 oracle.  The phase errors are float32 roundings of sums of
up to 65 terms and of two transforms, some 1e-7 of phases of up to ten
radians: rel. L2 < 5e-6."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs
from oracle import elasca_ref as E

from helpers import random_setup, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nats", [(16, 16, (1, 0)), (48, 32, (31, 33)), (64, 96, (32, 65)), (625, 48, (33,)),
                                        (160, 320, (0, 64, 5)), (512, 512, (33, 1, 32, 0, 65, 7, 40, 31)),
                                        (640, 625, (32, 33, 20, 1, 50, 65))])
@pytest.mark.parametrize("bwl", [False, True])
def test_formfactor_tiles(nx, ny, nats, bwl):
    a, b, cz = 0.02 * nx, 0.02 * ny, 0.2
    nvar = len(nats)
    sp = random_setup(nx, ny, nslices=1, nvar=(nvar, nvar), seed=3)
    sp = configs.Setup(**{**sp.__dict__, "a0": (a, b, cz)})
    rng = np.random.default_rng(nx + ny)
    q2 = E.freqs(nx, a).astype(np.float64)[None, :] ** 2 + E.freqs(ny, b).astype(np.float64)[:, None] ** 2
    ff = np.stack([amp * np.exp(-2 * np.pi ** 2 * s * s * q2) * (1 + 1j * ab)
                   for s, amp, ab in ((0.015, 25.0, 0.05), (0.05, 40.0, 0.08), (0.08, 70.0, 0.0))]).astype(np.complex64)
    sets = []
    for v, k in enumerate(nats):
        xy = np.stack([rng.uniform(-0.3, a + 0.3, k), rng.uniform(-0.3, b + 0.3, k)], 1).astype(np.float32)
        typ = (2 * rng.integers(0, 2, k) if v % 2 else rng.integers(0, 3, k)).astype(np.int32)
        sets.append((xy, typ, rng.uniform(0.5, 1.0, k).astype(np.float32)))
    eng = Engine().setup(sp)
    eng.formfactor_gratings(0, ff, sets, cz, bwl_pot=bwl, bwl_pgr=bwl)
    dev = eng.gratings(0, nvar)
    eng.close()
    for v, (xy, typ, occ) in enumerate(sets):
        ref = E.phase_grating(nx, ny, a, b, cz, sp.wl, ff, xy, typ, occ, bwl_pot=bwl, bwl_pgr=bwl)
        e = rel_l2(dev[v], ref)
        print(f"variant {v}, {len(occ)} atoms: {e:.2e}")
        assert e < 5e-6
