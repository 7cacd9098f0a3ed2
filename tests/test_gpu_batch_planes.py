"""Four phi planes per thread in a batch: chosen where they are the faster kernel (many blocks, few BC
blocks, the radiation BC, no member on other planes) and nowhere else, and with members of 4 and of more
planes in one launch the states are bit for bit those of the one-substep kernel."""
import numpy as np
import pytest

from nrpyelliptic_amd import config, runtime

pytestmark = pytest.mark.gpu


def problems(grids):
    probs = [runtime.Problem(config.random_batch(1, seed=k, grids=False, Nxx=n)[0]) for k, n in enumerate(grids)]
    for P in probs:
        P.set_wave_speed_cfl(0.5)
        P.zero_guess()
    return probs


BIG = [(128, 128, 16)] * 4  # 1024 four-plane blocks, 512 BC blocks


@pytest.mark.parametrize("grids,opts,want", [
    (BIG, {}, [4] * 4),
    (BIG, {"outer_bc": "sommerfeld6"}, [2] * 4),
    (BIG, {"tiles": [0, (32, 2), 0, 0]}, [2] * 4),              # a member asked for two planes
    (BIG, {"tiles": [0, 64, 0, 0]}, [2] * 4),                    # 64-wide tiles have two at most
    (BIG, {"tiles": [0, 16, 0, 0]}, [2, 1, 2, 2]),
    (BIG, {"substeps_per_launch": 1}, [2] * 4),
    (BIG + [(70, 18, 6)], {}, [2] * 5),                          # six planes: a launch of its own
    ([(160, 104, 16), (160, 104, 16)], {}, [2] * 2),             # 520 + 224 blocks: too few
    ([(32, 256, 32)] * 4, {}, [2] * 4),                          # 1024 and 2048 BC blocks
    ([(32, 128, 32), (40, 96, 16), (32, 200, 24)], {}, [2] * 3),
    ([(512, 256, 4), (256, 128, 8)], {}, [4] * 2),               # 768 + 128 blocks: the rule's limit
    (BIG * 3, {"outer_bc": "sommerfeld6"}, [4] * 12),            # 4608 blocks: either BC
    (BIG * 3 + [(70, 18, 6)], {}, [4] * 12 + [2]),               # and beside another launch
    ([(96, 128, 16)] * 5, {}, [2] * 5),                          # 960 + 640, BC blocks two thirds
    ([(96, 128, 16)] * 7, {}, [4] * 7),                          # 1344 + 896: enough blocks for that share
    ([(512, 256, 4), (256, 120, 8)], {}, [2] * 2),               # 752 + 128: below it
], ids=lambda v: str(v)[:40])
def test_planes_chosen(grids, opts, want):
    probs = problems(grids)
    try:
        B = runtime.BatchSolver(probs, **opts)
        got = B.planes
        B.close()
        assert got == want
    finally:
        for P in probs:
            P.close()


@pytest.mark.parametrize("grids,any4", [([(512, 256, 4), (256, 128, 8), (200, 130, 16)], True),
                                        ([(512, 256, 4), (256, 128, 6), (40, 24, 2)], False),
                                        ([(128, 128, 16), (160, 96, 8), (128, 90, 12)] * 2, True),
                                        ([(128, 128, 16), (512, 128, 4)] * 6 + [(40, 24, 2)], None)])
@pytest.mark.parametrize("bc", ["radiation", "sommerfeld6"])
def test_states_equal_the_one_substep_kernel(grids, any4, bc):
    probs = problems(grids)
    try:
        want = []
        for P in probs:
            S = P.solver(max_steps=50, log10_target=-30.0, substeps_per_launch=1, outer_bc=bc)
            S.solve()
            S.close()
            want.append(P.get("y_n_gfs"))
            P.zero_guess()
        B = runtime.BatchSolver(probs, max_steps=50, log10_target=-30.0, outer_bc=bc)
        assert B.planes == [4 if any4 is None and n[2] % 4 == 0 or any4 and bc == "radiation" else 2 for n in grids]
        res, _ = B.solve()
        B.close()
        for P, w, r in zip(probs, want, res):
            assert r.steps == 50 and np.all(np.isfinite(w)) and np.array_equal(P.get("y_n_gfs"), w)
    finally:
        for P in probs:
            P.close()
