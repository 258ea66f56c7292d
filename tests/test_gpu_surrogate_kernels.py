"""The matrix-core kernels of the surrogate at the edges of their launches:
batches of one sample, fewer and more samples than compute units (a block
then works on several), ragged head blocks, and prediction chunks.  Samples
are independent, so outputs are compared bit for bit across batch shapes, and
the gradient of a batch with the mean of its halves' gradients (the 1 / n of
the loss is an exact factor of two between them, so the bf16 roundings agree
and only float32 summation orders differ: 1e-5 relative L2 is 80 times
float32's unit rounding)."""
import numpy as np
import pytest

from jmultislicelib_amd import surrogate as S
from oracle import surrogate_ref as R

from helpers import rel_l2

pytestmark = pytest.mark.gpu


def _windows(n, seed):
    rng = np.random.default_rng(seed)
    x = np.abs(rng.standard_normal((n, 8, 32, 32)) * 0.3).astype(np.float32)
    return S.bf16_bits(x), (rng.standard_normal((n, 3)) * 0.3).astype(np.float32)


@pytest.mark.parametrize("n", [1, 63, 255, 257, 700, 16385])
def test_predict_equals_forward(n):
    m = min(n, 700)
    xb, t = _windows(m, n)
    rep = np.resize(np.arange(m), n)
    net = S.Network(max_batch=256, seed=2)
    data = S.WindowSet.from_arrays(xb[rep], t[rep])
    got = net.predict(data)
    ref = np.concatenate([net.forward(xb[i:i + 100]) for i in range(0, m, 100)])
    assert np.array_equal(got, ref[rep])
    data.close()
    net.close()


@pytest.mark.parametrize("n", [2, 6, 130, 600])
def test_gradient_is_the_mean_of_the_halves(n):
    xb, t = _windows(n, n)
    sc = np.array([0.3, 0.1, 0.05], np.float32)
    net = S.Network(max_batch=n, seed=5)
    loss, g = net.gradients(xb, t, sc)
    h = n // 2
    (l1, g1), (l2, g2) = net.gradients(xb[:h], t[:h], sc), net.gradients(xb[h:], t[h:], sc)
    assert abs(loss - (l1 + l2) / 2) <= 1e-5 * abs(loss)
    o = 0
    for name, shape in R.layout():
        k = int(np.prod(shape))
        e = rel_l2(g[o:o + k], 0.5 * (g1[o:o + k].astype(np.float64) + g2[o:o + k]))
        assert e < 1e-5, f"{name}: {e:.2e}"
        o += k
    net.close()
