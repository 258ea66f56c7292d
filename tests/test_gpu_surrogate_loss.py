"""The loss of a training batch is summed in double: all parameters zero, so the
outputs are zero and the residuals are the targets; one sample of squared
residual 1 and the others 2^-25, which float32 additions one after the other
would drop.  Bound: three float32 roundings (a share's sum, the total or the
shares' sum, the quotient), 3 * 2^-24; the dropped part is 15 * 2^-25 of the sum
or more."""
import numpy as np
import pytest

from jmultislicelib_amd import surrogate as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256, 1000])
def test_loss_in_double(n):
    t = np.full((n, 3), 2.0 ** -13, np.float32)
    t[:, 2] = 0
    t[0] = (1, 0, 0)
    want = (1 + (n - 1) * 2.0 ** -25) / (3 * n)
    net = S.Network(max_batch=n, seed=1)
    net.set_params(np.zeros(net.num_params(), np.float32))
    x = np.zeros((n, 8, 32, 32), np.uint16)
    loss, _ = net.gradients(x, t, np.ones(3, np.float32))
    net.close()
    assert abs(float(loss) - want) <= 3 * 2.0 ** -24 * want, f"{loss:.9e} for {want:.9e}"
