"""The allocation-free entry at 625-point columns: its waves lie in the natural
layout, in 16-column tiles, so a batch of up to 4 Mi readout sums in those tiles
is taken (the 8-column tiles of the panels would need up to twice as many).
Sums against the staged scan of the same inputs, which takes the panels: the
same transforms, sums over the columns in another order, so within 1e-6 of the
largest value (20 times float32's unit rounding)."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs

from helpers import random_setup
from test_zz_no_alloc import _Hip, _noalloc

pytestmark = pytest.mark.gpu
RINGS = tuple((4.0 * k, 4.0 * k + 6.0) for k in range(8))
SCRATCH = 4 << 20  # floats


@pytest.mark.parametrize("nx,slices,waves", [(16, 64, 5000), (48, 7, 40), (640, 3, 5), (625, 4, 6)])
def test_wide_tiles(nx, slices, waves):
    sp = random_setup(nx, 625, nslices=slices, nvar=(2, 1), ndetper=1, seed=nx, det_ranges=RINGS)
    per = waves * (slices + 1) * len(RINGS)
    assert per * -(-nx // 16) <= SCRATCH and (nx > 16 or per * -(-nx // 8) > SCRATCH)
    rng = np.random.default_rng(nx)
    dx, dy = rng.uniform(0, 0.15, (2, waves)).astype(np.float32)
    var = configs.variant_sequences(sp, waves, seed=3)
    w = np.ones(1, np.float32)
    eng = Engine().setup(sp)
    got = _noalloc(eng, _Hip(), waves, 1, dx, dy, w, var)
    eng.stage_scan(dx, dy, None, w, var)
    eng.run_staged(0, waves)
    eng.sync()
    want = eng.scan_results()
    eng.close()
    assert np.abs(got - want).max() <= 1e-6 * np.abs(want).max()
