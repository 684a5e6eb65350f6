"""Both transforms of a small plane in one launch (planes of at most 64 x 64) where it can go wrong:
the tiniest planes, one past a tile of 16 outputs or a step of 8 inputs on either axis, the largest
planes and the first size past them (line kernels), every pair of transform kinds, with and without
z tiles, against the oracle; and as members of one batch, bitwise the single solves.

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

KINDS = ["PP", "NN", "DD", "ND", "DN"]
# (the oracle, like the reference, takes periodic x with periodic y only)
PAIRS = [a + b for a in KINDS for b in KINDS if a != "PP" or b == "PP"]
PLANES = [(2, 2), (2, 64), (64, 2), (3, 17), (15, 16), (17, 15), (16, 33), (31, 7), (24, 20), (49, 48), (63, 64),
          (64, 63), (64, 64), (65, 64), (64, 65)]
BOX = [-0.25, 1.0, 0.0, 1.5, 0.0, 0.5]


def _case(i, nx, ny, pair):
    zbc, nz = [("DD", 9), ("NN", 18), ("PP", 16), ("DN", 33)][i % 4]
    return (nz, ny, nx), pair + zbc


@pytest.mark.parametrize("pair", PAIRS)
def test_plane_matches_oracle(pair):
    for i, (nx, ny) in enumerate(PLANES):
        shape, bc = _case(i + PAIRS.index(pair), nx, ny, pair)
        print(f"plane {bc} {shape}", flush=True)
        f = prng.uniform_pm1(shape, seed=nx + ny)
        ref = oracle.solve(f, bc, BOX, zero_mode=1)
        for zlayout in (1, 0):
            got = pa.solve(f, bc, BOX, zero_mode=1, zlayout=zlayout)
            err = float(np.abs(got - ref).max() / np.abs(ref).max())
            assert err <= 1e-12, f"{bc} {shape} zlayout={zlayout}: rel max diff {err:.3e}"


def test_plane_batch_is_the_single_solves():
    cases = [_case(i, nx, ny, PAIRS[(5 * i) % len(PAIRS)]) for i, (nx, ny) in enumerate(PLANES)]
    rhs = [prng.uniform_pm1(shape, seed=i) for i, (shape, _) in enumerate(cases)]
    with pa.Batch() as B:
        for shape, bc in cases:
            B.add(shape[2], shape[1], shape[0], bc, BOX)
        B.finalize()
        for i, f in enumerate(rhs):
            B.set_rhs(i, f)
        B.solve()
        for i, ((shape, bc), f) in enumerate(zip(cases, rhs)):
            print(f"batch member {bc} {shape}", flush=True)
            one = pa.solve(f, bc, BOX)
            assert np.array_equal(B.get_solution(i), one), f"member {i} {bc} {shape}"
