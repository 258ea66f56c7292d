"""Batches whose waves go through the slices in parts that stay in the Infinity
Cache, each part in two halves on two streams: the same scan in small batches
(one stream, one part) computes the same sums.  The shapes' instantiations may
contract products differently: 1e-6 of the largest value, as between the
band-limited and the general path."""
import numpy as np
import pytest

from jmultislicelib_amd import Engine, configs

from helpers import random_setup

pytestmark = pytest.mark.gpu
TOL = 1e-6


# waves: odd and even counts, below and above what two halves ask for (40 MiB
# stored), one part and several (184 MiB less the gratings), and waves too
# large for parts (10 of 2048^2: streamed; 3 of them: two unequal halves)
@pytest.mark.parametrize("nx,ny,nwave", [(160, 160, 1601), (256, 256, 101), (256, 256, 130), (256, 256, 561),
                                         (256, 512, 129), (360, 320, 97), (512, 512, 49), (512, 512, 320),
                                         (625, 640, 45), (720, 720, 62), (1024, 1024, 41), (2048, 2048, 3),
                                         (2048, 2048, 10), (96, 1024, 201)])
def test_parts_equal_small_batches(nx, ny, nwave):
    sp = random_setup(nx, ny, nslices=3, nvar=(2, 2), ndetper=2, seed=nx + 5 * ny)
    npass = 2 if nwave % 2 == 0 else 1
    npos = nwave // npass
    rng = np.random.default_rng(nwave)
    dx, dy = rng.uniform(0, 0.4, (2, npos)).astype(np.float32)
    var = configs.variant_sequences(sp, nwave, seed=6)
    w = np.full(npass, 1.0 / npass, np.float32)
    small = max(npass, (8 << 20) // (8 * nx * ny) // npass * npass)
    eng = Engine().setup(sp)
    got = {}
    for batch, graph in ((small, False), (0, False), (0, True)):
        eng.set_batch(batch)
        eng.set_graph(graph)
        for islc0 in (0, 2):
            eng.stage_scan(dx, dy, None, w, var)
            for _ in range(3 if graph else 1):  # replays with other work between
                eng.run_staged(0, npos, islc0)
                eng.sync()
            got[batch, graph, islc0] = eng.scan_results()
    eng.close()
    for (batch, graph, islc0), r in got.items():
        ref = got[small, False, islc0]
        d = np.abs(r - ref).max() / np.abs(ref).max()
        assert d <= TOL, f"batch {batch}, graph {graph}, from plane {islc0}: {d:.2e}"
