"""The drop-in calls return as soon as a flag behind their kernels is seen in host memory, without a
runtime synchronisation. Everything they wrote must then be complete for any reader: a copy or a kernel
on another stream that no runtime call has ordered behind the library's work, and several host threads
calling at once. Bar: bit-identical to the same calls each followed by a device synchronisation."""
import concurrent.futures as cf
import ctypes as C

import numpy as np
import pytest
import torch

from nrpyelliptic_amd import abi, config, runtime

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16, 6), (64, 48, 16), (200, 130, 16)]


class Buffer:
    """A tensor's view of one of a problem's device buffers; the problem outlives it."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(C.cast(ptr, C.c_void_p).value, False),
                                             version=2, strides=None)


def run_calls(shape, seed, sync):
    """Every short call on one problem, its output read on another stream right after it."""
    P = runtime.Problem(config.shipped_free_parameters(shape))
    L, p, gf, out = runtime.lib(), P.gd.params, P.gd.gridfuncs, []
    side = torch.cuda.Stream()
    y, k = (torch.as_tensor(Buffer(q, 2 * P.ntot), device="cuda") for q in (gf.y_n_gfs, gf.k_odd_gfs))
    res = torch.as_tensor(Buffer(gf.diagnostic_output_gfs, P.ntot), device="cuda")
    ws = (C.c_double * 2)(p.uu_wavespeed_at_OB, p.vv_wavespeed_at_OB)
    finf = (C.c_double * 2)(0.0, 0.0)

    def read(t):
        if sync:
            torch.cuda.synchronize()
        with torch.cuda.stream(side):
            by_kernel = t * 2.0
            out.append(t.cpu().numpy())
            out.append(by_kernel.cpu().numpy())

    try:
        P.set("y_n_gfs", 1e-3 * np.random.default_rng(seed).standard_normal(2 * P.ntot))
        P.set("k_odd_gfs", np.zeros(2 * P.ntot))
        for _ in range(4):
            L.rhs_eval(C.byref(p), C.byref(P.gd.rfmstruct), gf.auxevol_gfs, gf.y_n_gfs, gf.k_odd_gfs)
            read(k)
            L.apply_bcs_outerradiation_and_inner(C.byref(p), C.byref(P.gd.bcstruct), P.gd.xx, C.byref(ws),
                                                 C.byref(finf), gf.y_n_gfs, gf.k_odd_gfs)
            read(k)
            P.mol_step()
            read(y)
            L.apply_bcs_inner_only(C.byref(p), C.byref(P.gd.bcstruct), gf.y_n_gfs)
            read(y)
            L.residual_all_points(C.byref(p), C.byref(P.gd.rfmstruct), gf.auxevol_gfs, gf.y_n_gfs,
                                  gf.diagnostic_output_gfs)
            read(res)
            out.append(np.array([L.L2_norm_of_gf(C.byref(p), abi.UUGF, 100.0, P.gd.xx, gf.diagnostic_output_gfs)]))
        torch.cuda.synchronize()
        del y, k, res
    finally:
        P.close()
    return out


def same(a, b):
    return len(a) == len(b) and all(np.array_equal(x, v, equal_nan=True) for x, v in zip(a, b))


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_outputs_are_complete_on_other_streams(shape):
    want = run_calls(shape, 1, True)
    for _ in range(3):
        assert same(run_calls(shape, 1, False), want)


def test_outputs_are_complete_with_several_threads():
    want = [run_calls(SHAPES[k % 2], k, True) for k in range(4)]
    with cf.ThreadPoolExecutor(4) as ex:
        got = list(ex.map(lambda k: run_calls(SHAPES[k % 2], k, False), range(4)))
    for k in range(4):
        assert same(got[k], want[k]), k
