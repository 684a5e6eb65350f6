"""pp_solve_device_oop_noalloc where the dense-product matrices of one axis do not fit its device array:
that axis runs as the chirp convolution, the others keep their products; grids whose matrices all fit,
before and after, rebuild the tables.

Bars: bitwise the handle in place without Thomas columns where all matrices fit; else max-norm difference
<= 1e-12 relative to max|u| of the handle and of the oracle, the FP64 bar of every parity test."""
import ctypes

import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

BOX = [0.0, 1.0, 0.0, 1.5, 0.0, 0.5]
# (nz, ny, nx), bc, do all matrices fit
CASES = [((31, 101, 97), "DDNNDD", True), ((97, 509, 101), "DDNNDD", False), ((9, 101, 97), "NNDDDN", True),
         ((40, 101, 509), "NNDDNN", True), ((12, 1021, 439), "NNNNDD", False), ((767, 64, 64), "NNNNPP", False),
         ((331, 101, 97), "PPPPPP", True)]


def test_axes_keep_the_products_that_fit():
    import torch

    L = pa.load_library()
    X = np.ascontiguousarray(BOX, dtype=np.float64)
    for i, (shape, bc, fits) in enumerate(CASES):
        print(f"noalloc axes {bc} {shape}", flush=True)
        nz, ny, nx = shape
        f = prng.uniform_pm1(shape, seed=60 + i)
        d_f = torch.from_numpy(f).cuda()
        d_u, d_v = torch.full_like(d_f, float("nan")), torch.empty_like(d_f)
        torch.cuda.synchronize()
        rc = L.pp_solve_device_oop_noalloc(nx, ny, nz, bc.encode(), X.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 1,
                                           d_f.data_ptr(), d_u.data_ptr(), torch.cuda.current_stream().cuda_stream)
        assert rc == 0, pa.error_name(rc)
        with pa.PoissonHIP(nx, ny, nz) as M:
            M.set_option(pa.OPT_ZLAYOUT, 0)
            M.set_option_double(pa.OPT_ZTHOMAS_TAU, 0.0)
            M.assignBoundary(bc)
            M.setBox(BOX)
            M.setCoords(2)
            torch.cuda.synchronize()
            M.solve_device_oop(d_f.data_ptr(), d_v.data_ptr())
            torch.cuda.synchronize()
        u, v = d_u.cpu().numpy(), d_v.cpu().numpy()
        if fits:
            assert np.array_equal(u, v), (shape, bc)
        assert np.abs(u - v).max() <= 1e-12 * np.abs(v).max(), (shape, bc)
        ref = oracle.solve(f, bc, BOX, zero_mode=1)
        assert np.abs(u - ref).max() <= 1e-12 * np.abs(ref).max(), (shape, bc)
