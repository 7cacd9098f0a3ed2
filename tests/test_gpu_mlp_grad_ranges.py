"""The gradient kernels on row counts that split differently over their 32 row ranges (steps per
range not a multiple of the eight in flight, a short last range, empty ranges, the production
minibatch), against the FP64 restatement with the tolerances of the gradient test beside it; and
the training step's fused Adam against a gradient call followed by an Adam call on the same rows:
the same sums and the same update, so the weights are equal bit for bit."""
import numpy as np
import pytest

from nrpyelliptic_amd import mlp as nmlp
from nrpyelliptic_amd.runtime import DeviceArray, check
from oracle import mlp_ref

pytestmark = pytest.mark.gpu


def dataset(N, seed):
    rng = np.random.default_rng(seed)
    X = np.zeros((N, nmlp.K0), np.float32)
    X[:, :23] = rng.uniform(-1, 1, (N, 23))
    bits = nmlp.bf16_bits(X).reshape(N, nmlp.K0)
    return bits, rng.uniform(-1, 1, N).astype(np.float32)


# ranges x steps: 23 ranges of 3 (the last 2), 29 of 9 (the last 8), 32 of 16
@pytest.mark.parametrize("M", [1088, 4160, 8192])
def test_gradients_over_row_ranges(M):
    net = nmlp.InitialGuessMLP(seed=21)
    p = net.get_params().astype(np.float64)
    bits, t = dataset(M, M)
    loss, g = net.loss_grad(DeviceArray(bits.size, np.uint16).upload(bits.ravel()), DeviceArray(M, np.float32).upload(t), M)
    loss_ref, g_ref = mlp_ref.loss_grad(p, nmlp.bf16_to_float(bits).astype(np.float64), t.astype(np.float64))
    assert loss == pytest.approx(loss_ref, rel=1e-3)
    off = 0
    for l in range(1, 6):
        for size in (256 * (64 if l == 1 else 256), 256):
            a, b = g[off:off + size], g_ref[off:off + size]
            assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b) + 1e-12, (l, size)
            off += size
    assert np.linalg.norm(g[off:] - g_ref[off:]) <= 1e-2 * np.linalg.norm(g_ref[off:])


@pytest.mark.parametrize("M", [64, 1088, 8192])
def test_fused_adam_equals_gradient_then_adam(M):
    N, seed, lr = 3000, 9, np.float32(1e-3)
    bits, t = dataset(N, 4)
    z = np.arange(1, M + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)  # the library's row draw of step 0
    z += np.uint64((seed + 0x632BE59BD9B4E019) & ((1 << 64) - 1))
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    rows = ((z ^ (z >> np.uint64(31))) % np.uint64(N)).astype(np.int64)
    a, b = nmlp.InitialGuessMLP(seed=5), nmlp.InitialGuessMLP(seed=5)
    a.train(DeviceArray(bits.size, np.uint16).upload(bits.ravel()), DeviceArray(N, np.float32).upload(t), N, M, 1,
            float(lr), seed)
    xb, tb = bits[rows], t[rows]
    b.loss_grad(DeviceArray(xb.size, np.uint16).upload(xb.ravel()), DeviceArray(M, np.float32).upload(tb), M)
    first = lr * (np.float32(0.01) + np.float32(0.99) * np.float32(0.5) * np.float32(2.0))
    check(nmlp._bind().nrpyell_mlp_adam_step(b.h, float(first)), "adam_step")
    assert np.array_equal(a.get_params(), b.get_params())
