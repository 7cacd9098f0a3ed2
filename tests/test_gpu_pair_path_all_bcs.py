"""The two-substep kernel with the thorn's Sommerfeld outer BC and on grids with 2 and 4 phi planes
(a phi window longer than the period) against the one-substep kernel: bit-identical states, for
every tile shape, on ragged grids, Nxx1 from the smallest allowed (10) past the BC blocks' 16 rows,
in FP32 bulk solves and in batches. The one-substep kernel follows the oracle for both BCs
(test_gpu_sommerfeld.py, test_gpu_parity.py)."""
import numpy as np
import pytest

from nrpyelliptic_amd import config, runtime

pytestmark = pytest.mark.gpu

CASES = [((16, 16, 6), "sommerfeld6"), ((33, 16, 6), "sommerfeld6"), ((70, 12, 6), "sommerfeld6"),
         ((40, 36, 8), "sommerfeld6"), ((64, 64, 4), "radiation"), ((64, 64, 4), "sommerfeld6"),
         ((24, 12, 2), "radiation"), ((24, 12, 2), "sommerfeld6"), ((45, 10, 4), "radiation"),
         ((45, 10, 4), "sommerfeld6")]
TILES = [(32, 1), (16, 1), (64, 1), (32, 2), (64, 2)]


@pytest.fixture(scope="module", params=CASES, ids=lambda c: "x".join(map(str, c[0])) + "-" + c[1])
def prob(request):
    Nxx, bc = request.param
    P = runtime.Problem(config.random_batch(1, seed=3, grids=False, Nxx=Nxx)[0])
    P.set_wave_speed_cfl(0.5)
    yield P, bc
    P.close()


def steps(P, bc, n, spl, tile):
    P.zero_guess()
    S = P.solver(substeps_per_launch=spl, outer_bc=bc, tile_i0=tile[0], planes=tile[1])
    assert S.substeps_per_launch == (1 if spl == 1 else 2)
    S.steps(n)
    S.close()
    return P.get("y_n_gfs")


@pytest.mark.parametrize("tile", TILES, ids=lambda t: f"tx{t[0]}_pl{t[1]}")
def test_default_path_equals_one_substep(prob, tile):
    P, bc = prob
    for n in (1, 2, 31):
        a, b = steps(P, bc, n, 1, tile), steps(P, bc, n, 0, tile)
        assert np.all(np.isfinite(a))
        assert np.array_equal(a, b), (n, float(np.max(np.abs(a - b))))


def test_fp32_bulk_and_batch_equal_one_substep(prob):
    P, bc = prob
    out = []
    for spl in (1, 0):
        P.zero_guess()
        S = P.solver(substeps_per_launch=spl, outer_bc=bc, precision=32, max_steps=100, log10_target=-30.0,
                     fp32_switch_log10=-30.0)
        r = S.solve()
        out.append((r.steps, r.fp32_steps, P.get("y_n_gfs")))
        S.close()
    assert out[0][:2] == out[1][:2] and np.array_equal(out[0][2], out[1][2])
    P.zero_guess()
    S = P.solver(substeps_per_launch=1, outer_bc=bc, max_steps=100, log10_target=-30.0)
    S.solve()
    want = P.get("y_n_gfs")
    S.close()
    P.zero_guess()
    B = runtime.BatchSolver([P], outer_bc=bc, max_steps=100, log10_target=-30.0)
    B.solve()
    B.close()
    assert np.array_equal(P.get("y_n_gfs"), want)
