"""Initialize_ADMBase on a grid of more than 2^32 points (2048 x 2048 x 1100 with ghosts, 36.9 GB per
gridfunction): the molecules of points in the last phi planes start beyond the reach of a 32-bit index.
u = xx2 is a polynomial that every order reproduces, so uuGF must be the point's own phi. Bar 2e-12:
7^3 products of a value below pi with weights whose absolute sum is below 12, one rounding each."""
import ctypes as C

import numpy as np
import pytest
import torch

from nrpyelliptic_amd import abi, config, runtime
from nrpyelliptic_amd.runtime import ADMBASE_NAMES, DeviceArray

pytestmark = pytest.mark.gpu

DIMS = (2048, 2048, 1100)


def test_points_beyond_32_bit_indices():
    P = runtime.Problem(config.shipped_free_parameters((16, 16, 6)))
    try:
        gd = abi.griddata_struct.from_buffer_copy(P.gd)
        lo, hi = (0.0, 0.0, -np.pi), (1.0, np.pi, np.pi)
        xx = []
        for d in range(3):
            n = DIMS[d] - 2 * abi.NGHOSTS
            xx.append(lo[d] + (np.arange(DIMS[d]) - abi.NGHOSTS + 0.5) * ((hi[d] - lo[d]) / n))
            setattr(gd.params, f"Nxx{d}", n)
            setattr(gd.params, f"Nxx_plus_2NGHOSTS{d}", DIMS[d])
            gd.xx[d] = xx[d].ctypes.data_as(abi.REALP)
        plane = DIMS[0] * DIMS[1]
        assert plane * DIMS[2] > 1 << 32
        u = torch.empty(plane * DIMS[2] + plane, dtype=torch.float64, device="cuda")
        u[: plane * DIMS[2]].view(DIMS[2], plane).copy_(torch.from_numpy(xx[2]).cuda()[:, None].expand(-1, plane))
        torch.cuda.synchronize()
        gd.gridfuncs.y_n_gfs = C.cast(u.data_ptr(), abi.REALP)
        # half of the points below plane 1024, half above it
        phi = np.concatenate([np.linspace(-3.0, 2.6, 40), np.linspace(2.8, 3.12, 40)])
        pts = [DeviceArray(phi.size).upload(v) for v in (7.0 * np.cos(phi), 7.0 * np.sin(phi), np.linspace(-9, 9, 80))]
        outs = [DeviceArray(phi.size) for _ in ADMBASE_NAMES]
        o = runtime.admbase_options()
        o.orbital_plane, o.lapse_exponent_n, o.NRPy_epsilon = 1, -2.0, 1e-8
        for order in (1, 4, 6):
            o.interpolation_order = order
            rc = runtime.lib().nrpyell_Initialize_ADMBase(C.byref(gd), C.byref(o), (C.c_int * 3)(phi.size, 1, 1),
                                                          *[d.as_real_p() for d in pts], *[d.as_real_p() for d in outs])
            assert rc == 0, runtime.lib().nrpyell_last_error()
            assert np.max(np.abs(outs[0].download() - phi)) <= 2e-12, order
    finally:
        torch.cuda.synchronize()
        u = None
        torch.cuda.empty_cache()
        P.close()
