"""The two-substep kernel with four phi planes per thread, which the solvers choose by themselves where
its blocks make a full round (200x130x16: ragged in both directions; 256x128x16) and in batches:
the same states bit for bit as two planes per thread and as the one-substep kernel, in FP64, in the
FP32 bulk phase, in the drop-in step and in a batch."""
import numpy as np
import pytest

from nrpyelliptic_amd import config, runtime

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[(200, 130, 16), (256, 128, 16)], ids=lambda n: "x".join(map(str, n)))
def prob(request):
    P = runtime.Problem(config.random_batch(1, seed=3, grids=False, Nxx=request.param)[0])
    P.set_wave_speed_cfl(0.5)
    yield P
    P.close()


@pytest.mark.parametrize("bc", ["radiation", "sommerfeld6"])
def test_states_equal_other_tiles(prob, bc):
    out = []
    for opts in ({}, {"planes": 2}, {"substeps_per_launch": 1}):
        prob.zero_guess()
        S = prob.solver(outer_bc=bc, **opts)
        S.steps(7)
        out.append(prob.get("y_n_gfs"))
        prob.zero_guess()
        S.timed_steps(5)  # the fused residual check and the graph's odd tail
        out.append(prob.get("y_n_gfs"))
        for stage in (0, 1, 4) + ((5, 6) if S.substeps_per_launch == 2 else ()):
            assert S.time_substep(stage, 2) > 0.0
        S.close()
    assert np.all(np.isfinite(out[0]))
    for k in (2, 4):
        assert np.array_equal(out[0], out[k]) and np.array_equal(out[1], out[k + 1])


def test_residual_history_and_fp32(prob):
    out = []
    for opts in ({}, {"planes": 2}):
        prob.zero_guess()
        S = prob.solver(precision=32, max_steps=50, log10_target=-30.0, fp32_switch_log10=-30.0, **opts)
        r = S.solve()
        out.append((r.steps, r.fp32_steps, prob.get("y_n_gfs")))
        S.close()
        prob.zero_guess()
        S = prob.solver(max_steps=50, log10_target=-30.0, **opts)
        S.solve()
        out.append(S.history())
        S.close()
    assert out[0][:2] == out[2][:2] and np.array_equal(out[0][2], out[2][2])
    # the residual's partial sums follow the blocks: equal up to the order of 10^5 additions
    assert np.array_equal(out[1][0], out[3][0]) and np.max(np.abs(out[1][1] - out[3][1])) <= 1e-10


def test_drop_in_step(prob):
    prob.zero_guess()
    for _ in range(3):
        prob.mol_step()
    got = prob.get("y_n_gfs")
    prob.zero_guess()
    S = prob.solver(substeps_per_launch=1)
    S.steps(3)
    S.close()
    assert np.array_equal(got, prob.get("y_n_gfs"))


def test_batch():
    cfgs = [config.random_batch(1, seed=k, grids=False, Nxx=n)[0] for k, n in
            enumerate([(96, 96, 8), (128, 128, 16), (70, 18, 6)])]  # four planes, four planes, two (6 % 4)
    probs = [runtime.Problem(c) for c in cfgs]
    try:
        want = []
        for P in probs:
            P.set_wave_speed_cfl(0.5)
            P.zero_guess()
            S = P.solver(max_steps=50, log10_target=-30.0, planes=2)
            S.solve()
            want.append(P.get("y_n_gfs"))
            S.close()
            P.zero_guess()
        B = runtime.BatchSolver(probs, max_steps=50, log10_target=-30.0)
        res, _ = B.solve()
        B.close()
        for P, w, r in zip(probs, want, res):
            assert r.steps == 50 and np.array_equal(P.get("y_n_gfs"), w)
    finally:
        for P in probs:
            P.close()
