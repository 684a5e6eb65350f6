"""Line transforms as dense products on the matrix cores (lengths without a compiled plan) where
they can go wrong: one row or depth past a tile of 16 outputs or a step of 8 inputs, odd and even
middles, the tiniest lines, and both sides of the lengths (x 280, 440, 620, y 512) and of the numbers of
lines (2048, 3072 of more than 112 points) from which the chirp convolution takes over or gives way, for
every transform kind, against the oracle.

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

LENGTHS = [2, 3, 5, 13, 15, 17, 31, 34, 63, 65, 94, 129, 254, 257, 279, 281, 439, 441, 511, 513, 619, 621, 767, 1021]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("kind", ["PP", "NN", "DD", "ND", "DN"])
def test_dense_lines_match_oracle(kind, n):
    print(f"dense lines {kind} n={n}", flush=True)
    # (the oracle, like the reference, takes periodic x with periodic y only)
    shapes = [((5, 18, n), kind + ("PPDD" if kind == "PP" else "NNDD")), ((5, n, 18), "NN" + kind + "DN"),
              ((5, n, 17), "DD" + kind + "DD")]
    if n > 112:  # as many lines as it takes, and one row fewer
        rows = 64 if n <= 256 else 96
        shapes += [((rows, 32, n), shapes[0][1]), ((rows, n, 32), "NN" + kind + "DN"), ((rows - 1, n, 32), "DD" + kind + "DD")]
    for shape, bc in shapes:
        f = prng.uniform_pm1(shape, seed=n + len(bc))
        box = [-0.25, 1.0, 0.0, 1.5, 0.0, 0.5]
        ref = oracle.solve(f, bc, box, zero_mode=1)
        got = pa.solve(f, bc, box, zero_mode=1)
        err = float(np.abs(got - ref).max() / np.abs(ref).max())
        assert err <= 1e-12, f"{bc} {shape}: rel max diff {err:.3e}"
