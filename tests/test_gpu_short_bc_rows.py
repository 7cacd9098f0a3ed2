"""BC blocks of 8 rows, which the two-substep kernel has on grids whose blocks all run at once: the same
states bit for bit as its 16-row blocks (64-wide tiles have no others) and as the one-substep kernel, in
FP64, in the FP32 bulk phase and in the drop-in step. The grids: the smallest, one and two planes per
thread, rows that are no multiple of 8, and both sides of the rule's limits."""
import numpy as np
import pytest

from nrpyelliptic_amd import config, runtime

pytestmark = pytest.mark.gpu

GRIDS = [(10, 10, 2), (16, 16, 6), (64, 64, 4), (40, 60, 4), (64, 90, 8), (128, 64, 16), (128, 72, 16), (128, 128, 8)]


@pytest.fixture(scope="module", params=GRIDS, ids=lambda n: "x".join(map(str, n)))
def prob(request):
    P = runtime.Problem(config.random_batch(1, seed=5, grids=False, Nxx=request.param)[0])
    P.set_wave_speed_cfl(0.5)
    yield P
    P.close()


def states(prob, **opts):
    prob.zero_guess()
    S = prob.solver(**opts)
    S.steps(7)
    out = [prob.get("y_n_gfs")]
    prob.zero_guess()
    S.timed_steps(5)
    out.append(prob.get("y_n_gfs"))
    S.close()
    return out


@pytest.mark.parametrize("bc", ["radiation", "sommerfeld6"])
@pytest.mark.parametrize("planes", [0, 1, 2])
def test_states_equal_other_rows(prob, bc, planes):
    got = states(prob, outer_bc=bc, planes=planes)
    assert np.all(np.isfinite(got[0]))
    for opts in ({"tile_i0": 64, "planes": 1}, {"substeps_per_launch": 1}):
        want = states(prob, outer_bc=bc, **opts)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


def test_fp32_phase(prob):
    out = []
    for opts in ({}, {"tile_i0": 64, "planes": 1}):
        prob.zero_guess()
        S = prob.solver(precision=32, max_steps=50, log10_target=-30.0, fp32_switch_log10=-30.0, **opts)
        try:
            r = S.solve()
            out.append((r.steps, r.fp32_steps, prob.get("y_n_gfs")))
        except runtime.NrpyellError as e:  # 10x10x2 is too coarse to stay finite: it must be so on both
            out.append((str(e), "", np.zeros(1)))
        S.close()
    assert out[0][:2] == out[1][:2] and np.array_equal(out[0][2], out[1][2])


def test_drop_in_step(prob):
    prob.zero_guess()
    for _ in range(3):
        prob.mol_step()
    got = prob.get("y_n_gfs")
    prob.zero_guess()
    S = prob.solver(tile_i0=64, planes=1)
    S.steps(3)
    assert np.array_equal(got, prob.get("y_n_gfs"))
    S.close()


def test_short_blocks_are_chosen():
    P = runtime.Problem(config.random_batch(1, seed=5, grids=False, Nxx=(64, 64, 4))[0])
    S = P.solver()
    assert len(S.block_order()) == 4 * (2 * 8 + 8)  # one-plane interior blocks, 8-row BC blocks
    S.close()
    P.close()
