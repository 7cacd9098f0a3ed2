"""Solver.timed_steps takes every step it is asked for, also where the state diverges or becomes NaN on
the way: its time is that of n steps and its state that of n steps. Bar: bit-identical to Solver.steps,
which makes no residual check that could stop it."""
import numpy as np
import pytest

from nrpyelliptic_amd import config, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("substeps", [0, 1])
@pytest.mark.parametrize("n", [5, 60, 400])
def test_state_after_n_steps(n, substeps):
    P = runtime.Problem(config.random_batch(1, seed=3, grids=False, Nxx=(32, 24, 8))[0])
    try:
        P.set_wave_speed_cfl(1.2)  # above the stability limit: diverges within 400 steps
        S = P.solver(steps_per_graph=50, substeps_per_launch=substeps)
        P.zero_guess()
        S.steps(n)
        want = P.get("y_n_gfs")
        P.zero_guess()
        ms, l2 = S.timed_steps(n)
        got = P.get("y_n_gfs")
        steps, _ = S.history()
        S.close()
        assert ms > 0.0 and len(steps) == n
        if n == 400:
            assert not (np.max(np.abs(want)) < 1e12)  # it did diverge
        assert np.array_equal(got, want, equal_nan=True)
    finally:
        P.close()
