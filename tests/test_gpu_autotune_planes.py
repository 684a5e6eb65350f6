"""The autotuner on grids of small planes, whose x and y transforms run no line kernel: it tries none of
their shapes, so it reports the default shape of every line stage (which of several shapes it had picked
was timing noise), and the tuned solve matches the oracle.

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

PLANES = [(32, 32), (32, 24), (24, 32), (28, 32), (32, 20), (20, 32), (16, 32), (32, 16), (24, 24), (28, 28)]


@pytest.mark.parametrize("nx,ny", PLANES)
def test_no_line_shape_is_tuned(nx, ny):
    print(f"autotune plane {nx}x{ny}", flush=True)
    for nz, bc in ((40, "NNDDDD"), (96, "DDNNND"), (72, "DDDDNN")):
        f = prng.uniform_pm1((nz, ny, nx), seed=nz)
        ref = oracle.solve(f, bc, zero_mode=1)
        with pa.PoissonHIP(nx, ny, nz) as M:
            M.set_option(pa.OPT_AUTOTUNE, 1)
            M.assignBoundary(bc)
            M.setBox([0, 1, 0, 1, 0, 1])
            M.setCoords(2)
            M.assignRhs(f)
            M.pittPack()
            t = M.tuning()
            assert t["tuned"] and not any(t["line_variant"].values()), (nz, bc, t)
            got = M.getSolution()
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max(), (nz, bc)
