"""The fused inference kernel on row counts around its 64-row blocks and on weights set after the
network was made: the outputs follow the FP64 restatement that rounds where the kernel does
(oracle/mlp_ref.py). Tolerance: an activation whose FP32 value lies within FP32 rounding of a BF16
tie may round the other way, 2^-8 of it; at most a few of the 256 inputs of an output do, each
weighing 1/16 or so of it, as in the forward test at 256 rows."""
import numpy as np
import pytest

from nrpyelliptic_amd import mlp as nmlp
from nrpyelliptic_amd.runtime import DeviceArray
from oracle import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [64, 192, 64 * 257])  # one block; three; one more than the 256 CUs
def test_forward_rows_and_replaced_weights(M):
    net = nmlp.InitialGuessMLP(seed=1)
    rng = np.random.default_rng(M)
    p = (net.get_params() * rng.uniform(0.5, 1.5, net.n_params)).astype(np.float32)
    net.set_params(p)
    X = np.zeros((M, nmlp.K0), np.float32)
    X[:, :23] = rng.uniform(-1, 1, (M, 23))
    bits = nmlp.bf16_bits(X)
    y = net.forward(DeviceArray(bits.size, np.uint16).upload(bits.ravel()), M)
    y_ref, _, _ = mlp_ref.forward(p.astype(np.float64), nmlp.bf16_to_float(bits).astype(np.float64))
    assert np.max(np.abs(y - y_ref)) <= 5e-3 * np.max(np.abs(y_ref))
