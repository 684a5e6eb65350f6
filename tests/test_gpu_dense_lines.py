"""Line transforms as dense products on the matrix cores (lengths without a compiled plan) where
they can go wrong: one row or depth past a tile of 16 outputs or a step of 8 inputs, odd and even
middles, the tiniest lines, and both sides of the lengths from which the chirp convolution takes
over (x 340 / 620, y 512), for every transform kind, against the oracle.

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

LENGTHS = [2, 3, 5, 13, 15, 17, 31, 34, 63, 65, 94, 129, 254, 257, 339, 341, 511, 513, 619, 621, 767, 1021]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("kind", ["PP", "NN", "DD", "ND", "DN"])
def test_dense_lines_match_oracle(kind, n):
    print(f"dense lines {kind} n={n}", flush=True)
    # (the oracle, like the reference, takes periodic x with periodic y only)
    for shape, bc in (((5, 18, n), kind + ("PPDD" if kind == "PP" else "NNDD")), ((5, n, 18), "NN" + kind + "DN"),
                      ((5, n, 17), "DD" + kind + "DD")):
        f = prng.uniform_pm1(shape, seed=n + len(bc))
        box = [-0.25, 1.0, 0.0, 1.5, 0.0, 0.5]
        ref = oracle.solve(f, bc, box, zero_mode=1)
        got = pa.solve(f, bc, box, zero_mode=1)
        err = float(np.abs(got - ref).max() / np.abs(ref).max())
        assert err <= 1e-12, f"{bc} {shape}: rel max diff {err:.3e}"
