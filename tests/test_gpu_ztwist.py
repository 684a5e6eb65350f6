"""z columns of up to 128 rows, eliminated from both ends, where that can go wrong: the shortest, one row
past each 16 (an odd middle, a short last group of rows), the longest and the first past it, odd numbers of
16-column tiles, in place and on z tiles, every pair of z ends, both rules for the singular column,
nearly singular columns beside the others, and in a batch (bitwise the single solves).

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

ROWS = [4, 5, 15, 16, 17, 18, 31, 32, 33, 47, 63, 64, 65, 80, 81, 97, 112, 113, 127, 128, 129, 144]
BOX = [0.0, 1.0, 0.0, 1.5, -0.5, 0.5]


@pytest.mark.parametrize("nz", ROWS)
@pytest.mark.parametrize("zbc", ["DD", "NN", "DN", "ND"])
def test_columns_match_oracle(zbc, nz):
    for i, (nx, ny, xy) in enumerate([(17, 5, "NNNN"), (48, 3, "PPPP"), (16, 1 + nz % 2 + 1, "NDDN"), (130, 117, "NNNN")]):
        bc, shape = xy + zbc, (nz, ny, nx)
        print(f"z columns {bc} {shape}", flush=True)
        f = prng.uniform_pm1(shape, seed=nz + nx)
        for mode in (1, 0):
            if mode == 0 and (i or zbc == "NN"):
                continue  # the row-0 rule away from z NN: once
            ref = oracle.solve(f, bc, BOX, zero_mode=mode)
            for zlayout in (1, 0):
                got = pa.solve(f, bc, BOX, zero_mode=mode, zlayout=zlayout)
                err = float(np.abs(got - ref).max() / np.abs(ref).max())
                assert err <= 1e-12, f"{bc} {shape} zero_mode={mode} zlayout={zlayout}: rel max diff {err:.3e}"


def test_batched_columns_are_the_single_solves():
    cases = [((nz, 20 + nz % 3, 40), "DDNN" + ("NN" if nz % 2 else "DN")) for nz in ROWS] + [((33, 117, 130), "NNNNDN")]
    with pa.Batch() as B:
        for shape, bc in cases:
            B.add(shape[2], shape[1], shape[0], bc, BOX)
        B.finalize()
        rhs = [prng.uniform_pm1(shape, seed=i) for i, (shape, _) in enumerate(cases)]
        for i, f in enumerate(rhs):
            B.set_rhs(i, f)
        B.solve()
        for i, ((shape, bc), f) in enumerate(zip(cases, rhs)):
            print(f"batch member {bc} {shape}", flush=True)
            assert np.array_equal(B.get_solution(i), pa.solve(f, bc, BOX)), f"member {i} {bc} {shape}"
