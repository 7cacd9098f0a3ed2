"""The network seed's workspace over grids of different shapes: a long thin grid (more coordinates, fewer
rows than the one before) leaves the rows' arrays alone, so seeding the two grids in turn allocates once for
each. Seen from the free device memory: the rows' arrays of the larger grid, 40 MB, stay. The seeds are
those of a network that has seen no other grid."""
import numpy as np
import pytest
import torch

from nrpyelliptic_amd import config, runtime
from nrpyelliptic_amd import mlp as nmlp

pytestmark = pytest.mark.gpu


def test_grids_in_turn():
    probs = [runtime.Problem(config.random_batch(1, seed=k, grids=False, Nxx=n)[0])
             for k, n in enumerate([(128, 128, 16), (12, 12, 320)])]
    net = nmlp.InitialGuessMLP(seed=3)
    try:
        want = []
        for P in probs:
            fresh = nmlp.InitialGuessMLP(seed=3)
            fresh.seed(P, 2)
            want.append(P.get("y_n_gfs"))
            fresh.close()
        free = []
        for k in (0, 1, 0, 1, 0):
            net.seed(probs[k], 2)
            torch.cuda.synchronize()
            free.append(torch.cuda.mem_get_info()[0])
            assert np.array_equal(probs[k].get("y_n_gfs"), want[k])
        print(free)
        assert max(free[1:]) <= free[0] and min(free[1:]) == max(free[1:])
    finally:
        net.close()
        for P in probs:
            P.close()
