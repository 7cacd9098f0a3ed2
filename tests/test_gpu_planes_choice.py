"""Planes per thread of a solver that leaves them open: four where that is the faster kernel, in FP64 and in
FP32, and no more than two on either side of each limit; grids of four and of more planes give the states
of the one-substep kernel bit for bit with the four-plane kernel that is then known to run."""
import numpy as np
import pytest

from nrpyelliptic_amd import config, runtime

pytestmark = pytest.mark.gpu


def problem(n):
    P = runtime.Problem(config.random_batch(1, seed=3, grids=False, Nxx=n)[0])
    P.set_wave_speed_cfl(0.5)
    P.zero_guess()
    return P


# (four-plane blocks; BC blocks) on 256 CUs
@pytest.mark.parametrize("grid,fp64,fp32", [
    ((200, 130, 16), 4, 4),   # 476; 144
    ((256, 128, 16), 4, 4),   # 512; 128
    ((512, 256, 4), 4, 4),    # 512; 64
    ((224, 128, 16), 4, 4),   # 448; 128
    ((253, 108, 16), 4, 2),   # 448; 112: FP32 is better with two
    ((220, 120, 16), 2, 2),   # 420; 128: below the range
    ((96, 148, 32), 2, 2),    # 456; 320: just more than three blocks per CU in all
    ((93, 304, 16), 4, 4),    # 456; 304: three
    ((96, 160, 32), 2, 2),    # 480; 320
    ((64, 256, 32), 4, 4),    # 512; 512: two full rounds
    ((64, 232, 32), 2, 2),    # 464; 480
    ((32, 256, 64), 2, 2),    # 512; 1024
    ((256, 136, 16), 2, 2),   # 544; 144: beyond the range
    ((256, 256, 16), 4, 2),   # 1024; 256
    ((160, 192, 32), 2, 2),   # 960; 384: five tiles across
    ((123, 256, 32), 4, 2),   # 1024; 512
    ((32, 256, 128), 2, 2),   # 1024; 2048
    ((256, 288, 16), 4, 4),   # 1152; 288: FP32 from here on
    ((256, 256, 32), 4, 4),   # 2048; 512
    ((256, 256, 30), 2, 2),   # not a multiple of four planes
])
def test_planes_chosen(grid, fp64, fp32):
    P = problem(grid)
    try:
        for precision, want in ((64, fp64), (32, fp32)):
            S = P.solver(precision=precision)
            got = S.planes
            S.close()
            assert got == want, precision
        for opts, want in (({"planes": 2}, 2), ({"planes": 1}, 1), ({"tile_i0": 64}, 2), ({"tile_i0": 16}, 1)):
            S = P.solver(**opts)
            got = S.planes
            S.close()
            assert got == want, opts
    finally:
        P.close()


@pytest.mark.parametrize("grid", [(512, 256, 4), (256, 256, 8)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("bc", ["radiation", "sommerfeld6"])
def test_few_planes(grid, bc):
    P = problem(grid)
    try:
        out = []
        for opts, planes in (({}, 4), ({"planes": 2}, 2), ({"substeps_per_launch": 1}, 2)):
            P.zero_guess()
            S = P.solver(outer_bc=bc, **opts)
            assert S.planes == planes
            S.steps(6)
            out.append(P.get("y_n_gfs"))
            S.close()
        assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
        if bc == "radiation":
            P.zero_guess()
            for _ in range(2):
                P.mol_step()
            got = P.get("y_n_gfs")
            P.zero_guess()
            S = P.solver(substeps_per_launch=1)
            S.steps(2)
            S.close()
            assert np.array_equal(got, P.get("y_n_gfs"))
    finally:
        P.close()


@pytest.mark.parametrize("grid,bc_blocks,blocks", [((256, 128, 16), 128, 640), ((128, 256, 16), 256, 768),
                                                   ((256, 256, 32), 512, 0)])
def test_placement_with_four_planes(grid, bc_blocks, blocks):
    """Placed like the other kernels up to three blocks per CU: a permutation, the BC blocks first."""
    P = problem(grid)
    try:
        S = P.solver()
        assert S.planes == 4
        o = S.block_order()
        S.close()
        assert len(o) == blocks
        if blocks:
            assert np.array_equal(np.sort(o), np.arange(blocks)) and np.array_equal(o[:bc_blocks], np.arange(bc_blocks))
    finally:
        P.close()
