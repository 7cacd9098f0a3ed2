"""Initialize_ADMBase from several host threads: each call reports its own points' errors, also where more
calls are in flight than there are pinned flag lines (64) and the rest have theirs in device memory."""
import concurrent.futures as cf
import ctypes as C

import numpy as np
import pytest
import torch

from nrpyelliptic_amd import config, runtime
from nrpyelliptic_amd.runtime import ADMBASE_NAMES

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def prob():
    P = runtime.Problem(config.shipped_free_parameters((16, 16, 6)))
    P.set("y_n_gfs", 1e-3 * np.random.default_rng(0).standard_normal(2 * P.ntot))
    yield P
    P.close()


class Call:
    """A prepared call: its points, its outputs and the function to run on any thread."""

    def __init__(self, P, points):
        self.P, self.n = P, len(points)
        pts = torch.tensor(points, dtype=torch.float64, device="cuda").t().contiguous()
        self.pts, self.out = pts, torch.empty((len(ADMBASE_NAMES), self.n), dtype=torch.float64, device="cuda")
        self.o = runtime.admbase_options()
        self.o.lapse_exponent_n, self.o.NRPy_epsilon, self.o.interpolation_order = -2.0, 1e-8, 4
        torch.cuda.synchronize()

    def __call__(self):
        ptrs = [C.cast(t.data_ptr(), C.POINTER(C.c_double)) for t in (*self.pts, *self.out)]
        return runtime.lib().nrpyell_Initialize_ADMBase(C.byref(self.P.gd), C.byref(self.o),
                                                        (C.c_int * 3)(self.n, 1, 1), *ptrs)


def stall_ms(cycles):
    e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    e0.record()
    torch.cuda._sleep(cycles)
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1)


def calls_with_errors(prob, count):
    good = np.random.default_rng(2).normal(size=(200, 3)) * 8.0
    calls = []
    for k in range(count):
        X = good.copy()
        if k % 3 == 1:
            X[7] = np.nan
        if k % 3 == 2:
            X[9] = 1e9
        calls.append((Call(prob, X), (0, -5, -1)[k % 3]))
    return calls


def test_each_call_reports_its_own_errors(prob):
    calls = calls_with_errors(prob, 12)
    with cf.ThreadPoolExecutor(6) as ex:
        for _ in range(20):
            for (_, want), f in zip(calls, [ex.submit(c) for c, _ in calls]):
                assert f.result(60) == want


def test_more_calls_in_flight_than_flag_lines(prob):
    calls = calls_with_errors(prob, 80)
    for c, want in calls[:3]:
        assert c() == want
    per_ms = 1e8 / stall_ms(100_000_000)
    with cf.ThreadPoolExecutor(80) as ex:
        torch.cuda._sleep(int(300 * per_ms))  # every call is begun while the default stream is busy
        running = [ex.submit(c) for c, _ in calls]
        for (_, want), f in zip(calls, running):
            assert f.result(60) == want
    for c, want in calls[:3]:  # the lines came back
        assert c() == want
