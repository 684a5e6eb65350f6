"""Short periodic z in the one-pass kernel, whose blocks take as many columns as fill a wave, and 10 and 14
points, half a length of 5 or 7 held by one thread (no line transform of those lengths is compiled), where they
can go wrong: ragged x extents, with and without a singular column, every form, and a batch's members in one
launch of their class.

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test; batch
members bitwise the single solves."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48, 56, 80])
@pytest.mark.parametrize("nx", [16, 23, 70, 130])
def test_short_periodic_z(nx, nz):
    box = [0, 1, 0, 1, 0, nz / 16.0]
    for bc in ("PPPPPP", "DDNNPP", "NDDNPP"):
        print(f"short periodic z {bc} nx={nx} nz={nz}", flush=True)
        f = prng.uniform_pm1((nz, 6, nx), seed=nz + nx)
        ref = oracle.solve(f, bc, box)
        for zlayout, precision in ((0, 0), (1, 0), (1, 1)):
            got = pa.solve(f, bc, box, zlayout=zlayout, precision=precision)
            err = float(np.abs(got - ref).max() / np.abs(ref).max())
            assert err <= 1e-12, f"{bc} nz={nz} zlayout={zlayout} precision={precision}: {err:.3e}"


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nz", [10, 14, 16, 24, 48])
def test_short_periodic_z_members_share_a_launch(nz, precision):
    shapes = [(nz, 24, 24), (nz, 18, 23), (nz, 30, 66), (nz, 16, 16)]
    print(f"short periodic z batch nz={nz} precision={precision}", flush=True)
    with pa.Batch(precision=precision) as B:
        for s in shapes:
            B.add(s[2], s[1], s[0], "DDNNPP")
        B.finalize()
        assert B.launch_count()[2] == 1
        rhs = [prng.uniform_pm1(s, seed=i) for i, s in enumerate(shapes)]
        for i, f in enumerate(rhs):
            B.set_rhs(i, f)
        B.solve()
        for i, f in enumerate(rhs):
            assert np.array_equal(B.get_solution(i), pa.solve(f, "DDNNPP", precision=precision)), shapes[i]
