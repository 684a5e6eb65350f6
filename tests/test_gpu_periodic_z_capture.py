"""A caller's capture of the first FP64 solve of a handle whose tables an earlier mixed solve has built:
periodic z needs no second field, so the solve captures at every length, also from 512 rows, where solves
outside a capture hand the columns over in z tiles.

Bar: bitwise the solve outside the capture (both z layouts compute alike), on every replay."""
import numpy as np
import pytest

import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [384, 512, 640])
def test_capture_after_a_mixed_solve(nz):
    import torch

    print(f"capture periodic z nz={nz}", flush=True)
    f = prng.uniform_pm1((nz, 32, 48), seed=nz)
    ref = pa.solve(f, "NNDDPP")
    d_f = torch.from_numpy(f).cuda()
    d_u = torch.zeros_like(d_f)
    stream = torch.cuda.Stream()
    with pa.PoissonHIP(48, 32, nz) as M:
        M.assignBoundary("NNDDPP")
        M.setBox([0, 1, 0, 1, 0, 1])
        M.setCoords(2)
        M.set_option(pa.OPT_PRECISION, 1)
        M.set_stream(stream.cuda_stream)
        torch.cuda.synchronize()
        M.solve_device_oop(d_f.data_ptr(), d_u.data_ptr())
        torch.cuda.synchronize()
        M.set_option(pa.OPT_PRECISION, 0)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            M.solve_device_oop(d_f.data_ptr(), d_u.data_ptr())
        for replay in range(3):
            d_u.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(d_u.cpu().numpy(), ref), f"replay {replay}"
            M.solve_device_oop(d_f.data_ptr(), d_u.data_ptr())
            torch.cuda.synchronize()
            assert np.array_equal(d_u.cpu().numpy(), ref), f"eager {replay}"
