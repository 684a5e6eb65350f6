"""The one-pass periodic z solve where it can go wrong: the shortest and longest lengths, every
element count per thread, lengths past 512 (z tiles, 8-column blocks), x extents that leave a block
ragged, both z layouts, against the oracle.

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [8, 12, 20, 28, 64, 80, 96, 112, 320, 384, 512, 640, 768, 896, 1024])
@pytest.mark.parametrize("nx", [16, 23])
def test_periodic_z_one_pass(nx, nz):
    box = [0, 1, 0, 1, 0, nz / 16.0]
    for bc in ("PPPPPP", "DDNNPP"):
        print(f"periodic z {bc} nx={nx} nz={nz}", flush=True)
        f = prng.uniform_pm1((nz, 6, nx), seed=nz + nx)
        ref = oracle.solve(f, bc, box)
        for zlayout in (0, 1):
            got = pa.solve(f, bc, box, zlayout=zlayout)
            err = float(np.abs(got - ref).max() / np.abs(ref).max())
            assert err <= 1e-12, f"{bc} nz={nz} zlayout={zlayout}: {err:.3e}"
        got = pa.solve(f, bc, box, precision=1)
        err = float(np.abs(got - ref).max() / np.abs(ref).max())
        assert err <= 1e-12, f"{bc} nz={nz} mixed: {err:.3e}"
