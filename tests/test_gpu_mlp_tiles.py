"""The surrogate kernels at the edges of their tiles (32 samples in prediction,
64 in training) and with units far out or at zero, where silu and its
derivative are divided rather than taken from one reciprocal; against the
float64 oracle with the tolerances of test_gpu_mlp.py (BF16 operands agree up
to rare rounding flips, sums differ by FP32 rounding)."""
import numpy as np
import pytest

import muca_amd as M
from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


def _data(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (n, 4)).astype(np.float32)
    return x, np.sin(3 * x[:, 0]).astype(np.float32)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 65, 4097])
def test_prediction_tiles(n):
    p = MO.init_params(1)
    x, _ = _data(n, 2)
    with M.Mlp() as net:
        net.set_params(p)
        y, back = net.predict(x), net.predict(x[::-1])
    yr, _, _ = MO.forward_backward(p, x)
    top = max(1.0, np.max(np.abs(yr)))
    assert np.max(np.abs(y - yr)) <= 2e-3 * top
    assert np.array_equal(y, back[::-1])   # a sample's value does not depend on its place


@pytest.mark.parametrize("scale", [0.0, 60.0])
def test_gradient_of_zero_and_saturated_units(scale):
    """scale 0: every z1 and z2 is 0 (biases are); 60: most |z1| exceed 80."""
    p = MO.init_params(3)
    p[MO.OW1:MO.OB1] *= 4 * scale
    if scale:
        p[MO.OW2:MO.OB2] /= scale
    x, t = _data(130, 4)
    with M.Mlp() as net:
        net.set_params(p)
        g, loss = net.gradient(x, t)
    _, lr, gr = MO.forward_backward(p, x, t)
    assert np.isfinite(g).all() and abs(loss - lr) <= 1e-3 * abs(lr)
    assert np.linalg.norm(g - gr) <= 5e-3 * np.linalg.norm(gr)
