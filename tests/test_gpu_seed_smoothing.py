"""nrpyell_mlp_seed's smoothing against a NumPy restatement of it on the unsmoothed seed: passes
of (f[-1] + 2 f + f[+1]) / 4 along i0, i1, i2 over the interior, pure outer points kept, ghosts at
their parity images, v = eta u. The same IEEE operations in the same order: equal bit for bit.
Odd and even pass counts end in y_n through different buffers; the grids leave remainders in the
64-column blocks (and one of them two phi planes only); the feature rows are no multiple of the
feature kernel's 256-row blocks."""
import numpy as np
import pytest

from nrpyelliptic_amd import config, runtime
from nrpyelliptic_amd.mlp import InitialGuessMLP

pytestmark = pytest.mark.gpu
NG = 5


def pad(f):
    h = f.shape[0] // 2
    f = np.concatenate([np.roll(f[:, :, :NG][:, :, ::-1], h, 0), f], 2)
    f = np.concatenate([np.roll(f[:, :NG][:, ::-1], h, 0), f, np.roll(f[:, -NG:][:, ::-1], h, 0)], 1)
    return f[np.arange(-NG, f.shape[0] + NG) % f.shape[0]]


def smoothed(f, n0, passes):
    for _ in range(passes):
        for axis in (2, 1, 0):
            q = pad(f)
            c = [slice(NG, -NG)] * 3
            lo, hi = list(c), list(c)
            lo[axis], hi[axis] = slice(NG - 1, -NG - 1), slice(NG + 1, q.shape[axis] - NG + 1)
            f = f.copy()
            f[:, :, :n0] = 0.25 * (q[tuple(lo)] + q[tuple(hi)]) + 0.5 * q[tuple(c)]
    return f


@pytest.mark.parametrize("Nxx", [(33, 16, 6), (64, 12, 2), (60, 18, 8)])
def test_seed_smoothing_matches_numpy(Nxx):
    P = runtime.Problem(config.shipped_free_parameters(Nxx))
    net = InitialGuessMLP(seed=3)
    try:
        net.seed(P, 0)
        G = P.Ng[::-1]
        y0 = P.get("y_n_gfs").reshape(2, *G)
        eta = P.gd.params.eta_damping
        f0 = y0[0][NG:-NG, NG:-NG, NG:]
        assert np.array_equal(y0[0], pad(f0)) and np.array_equal(y0[1], eta * y0[0])
        for passes in (1, 2, 3):
            net.seed(P, passes)
            y = P.get("y_n_gfs").reshape(2, *G)
            want = pad(smoothed(f0, Nxx[0], passes))
            assert np.array_equal(y[0], want), passes
            assert np.array_equal(y[1], eta * want), passes
    finally:
        net.close()
        P.close()
