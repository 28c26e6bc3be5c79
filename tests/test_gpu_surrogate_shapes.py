"""The convolution kernels' block shapes: a batch large enough for the widest
blocks (four rows and every channel tile per wave) against one sample at a
time (one row, one channel tile), which the oracle covers.

The sum of an output runs over the same products in the same order in every
shape, so predictions are equal bit for bit.  A parameter gradient of n equal
samples is that of one sample up to the order of its FP32 sums: the bound of
the gradient tests against the oracle."""
import numpy as np
import pytest

from portlbm_amd import surrogate as sg

pytestmark = pytest.mark.gpu


def _inputs(B, H, W, seed):
    r = np.random.default_rng(seed)
    x = r.normal(size=(B, 4, H, W)).astype(np.float32)
    x[:, 0] = r.random(size=(B, H, W)) < 0.7
    return x, r.normal(size=(B, 3, H, W)).astype(np.float32)


# 240 x 272: remainders of rows and columns at every level below the first
@pytest.mark.parametrize("B,H,W", [(32, 256, 256), (34, 240, 272), (9, 16, 2048), (5, 1040, 16)])
@pytest.mark.parametrize("bf16", [False, True])
def test_predictions_do_not_depend_on_the_batch(B, H, W, bf16):
    x, _ = _inputs(B, H, W, 100 + H)
    with sg.Surrogate(H, W, max_batch=B) as net, sg.Surrogate(H, W, max_batch=1) as one:
        net.init_params(5)
        one.init_params(5)
        some = [0, B // 2, B - 1]
        whole = net.predict(x, bf16=bf16)[some]
        np.testing.assert_array_equal(whole, one.predict(x[some], bf16=bf16))


@pytest.mark.parametrize("B,H,W", [(32, 256, 256), (16, 240, 272), (5, 1040, 16)])
def test_gradient_of_equal_samples(B, H, W):
    x, t = _inputs(1, H, W, 200 + H)
    with sg.Surrogate(H, W, max_batch=B) as net:
        net.init_params(6)
        loss1, g1 = net.loss_grad(x, t)
        loss, g = net.loss_grad(np.repeat(x, B, axis=0), np.repeat(t, B, axis=0))
    assert loss == pytest.approx(loss1, rel=1e-5)
    assert np.linalg.norm(g - g1) <= 1e-4 * np.linalg.norm(g1)
