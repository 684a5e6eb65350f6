"""Short lines as dense products (up to 128 points; the other axis too long for the plane kernel, which
takes them otherwise): tile and depth edges, several lines a wave while they are staged along x,
quarter-wave lines along x from 2048 of them and the convolution one row below, for every transform kind,
in the FP64 form, as members of a batch, and against the oracle.

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test; members
bitwise the single solves."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from dense_line_shapes import KINDS, LENGTHS, shapes
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

BOX = [-0.25, 1.0, 0.0, 1.5, 0.0, 0.5]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("kind", KINDS)
def test_short_dense_lines(kind, n):
    cases = shapes(kind, n)
    rhs = [prng.uniform_pm1(shape, seed=n + i) for i, (shape, *_) in enumerate(cases)]
    with pa.Batch() as B:
        for shape, bc, *_ in cases:
            B.add(shape[2], shape[1], shape[0], bc, BOX)
        B.finalize()
        for i, f in enumerate(rhs):
            B.set_rhs(i, f)
        B.solve()
        for i, ((shape, bc, axis, _), f) in enumerate(zip(cases, rhs)):
            print(f"short dense lines {bc} {shape} axis {axis}", flush=True)
            ref = oracle.solve(f, bc, BOX, zero_mode=1)
            got = pa.solve(f, bc, BOX, zero_mode=1)
            err = float(np.abs(got - ref).max() / np.abs(ref).max())
            assert err <= 1e-12, f"{bc} {shape}: rel max diff {err:.3e}"
            assert np.array_equal(B.get_solution(i), got), (shape, bc)
