"""Solutions to host arrays by several threads through pinned chunks where it can go wrong: just below and
at the size from which it runs, whole and part chunks, odd counts, fewer chunks than threads, several
threads on one handle, and the serving form's copies; bytes are compared, not values."""
import threading

import numpy as np
import pytest

import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(128, 64, 63), (128, 64, 64), (129, 65, 63), (101, 97, 89), (128, 128, 128), (257, 129, 65)])
def test_solution_bytes(nx, ny, nz):
    print(f"host copy {nx}x{ny}x{nz}", flush=True)
    f = prng.uniform_pm1((nz, ny, nx), seed=nx)
    M = pa.PoissonHIP(nx, ny, nz)
    M.assignBoundary("NNDDDN")
    M.setBox([0, 1, 0, 1, 0, 1])
    M.setCoords(2)
    for _ in range(2):
        M.assignRhs(f)
        assert M.getSolution().tobytes() == f.tobytes()
    M.pittPack()
    once = M.getSolution().tobytes()
    got = [None] * 4

    def read(i):
        got[i] = M.getSolution().tobytes()

    threads = [threading.Thread(target=read, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(g == once for g in got)
    M.close()


@pytest.mark.parametrize("shape", [(16, 16, 16), (65, 63, 129), (64, 128, 128)])
def test_served_solution_bytes(shape):
    print(f"served host copy {shape}", flush=True)
    f = prng.uniform_pm1(shape, seed=5)
    nz, ny, nx = shape
    with pa.Batch() as B:
        B.add(nx, ny, nz, "NNDDDN", [0, 1, 0, 1, 0, 1])
        B.finalize()
        B.set_rhs(0, f)
        B.solve()
        ref = B.get_solution(0).tobytes()
    S = pa.Server(hbm_bytes=1 << 30, staging_bytes=1 << 28, streams=2)
    tickets = [S.submit(shape, "NNDDDN", rhs=f) for _ in range(3)]
    assert all(S.wait(t)[0].tobytes() == ref for t in tickets)
