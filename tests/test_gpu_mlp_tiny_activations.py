"""Activations of large negative inputs, whose sigmoid is a denormal FP32 number (z below -87.3): they are
not flushed to zero. The last hidden layer's inputs are its biases (its weights are zero) and one output
weight of 1e36 brings z sigmoid(z) into range. Bar: the activation is the BF16 number nearest to the FP64
value (none of the inputs lies within 1e-4 of a rounding tie, relatively; the FP32 evaluation is good to
1e-5), the output its FP32 product; beyond the exponential's range (z below -88.7) both are 0."""
import numpy as np
import pytest

from nrpyelliptic_amd import mlp as nmlp
from nrpyelliptic_amd.runtime import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("z", [-0.5, -20.0, -87.0, -87.3, -87.4, -88.0, -88.5, -88.6, -89.0, -200.0])
def test_denormal_sigmoids(z):
    net = nmlp.InitialGuessMLP(seed=1)
    M, W, n = 64, nmlp.WIDTH, net.n_params
    scale = np.float32(1e36 if z < -80.0 else 1.0)
    z32 = float(np.float32(z))
    p = np.zeros(n, np.float32)
    p[n - 1 - 2 * W + 3], p[n - 1 - W + 3] = z32, scale  # b_5 and the output weight of unit 3
    net.set_params(p)
    h = z32 / (1.0 + np.exp(-z32)) if z32 > -88.72 else 0.0
    want = nmlp.bf16_to_float(nmlp.bf16_bits(np.array([h], np.float32)))[0] * scale
    x = DeviceArray(M * nmlp.K0, np.uint16).upload(np.zeros(M * nmlp.K0, np.uint16))
    t = DeviceArray(M, np.float32).upload(np.zeros(M, np.float32))
    y = net.forward(x, M)
    loss, _ = net.loss_grad(x, t, M)  # the training forward pass: (y - 0)^2
    print(z, y[0], want, loss)
    assert np.all(np.abs(y - want) <= 2.0 ** -23 * abs(want))
    assert abs(loss - float(want) ** 2) <= 2.0 ** -20 * float(want) ** 2
