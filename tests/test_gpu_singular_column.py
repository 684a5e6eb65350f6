"""The singular (0, 0) column by scans over 64 lanes of ceil(nz / 64) rows: the shortest columns,
one row past a lane's share, and 1024 rows, periodic z (FP64, mixed, batched) and the mixed form's
pinned column with Neumann and (zero mode 0) Dirichlet last rows, against the oracle.

Bar: max-norm difference <= 1e-12 relative to max|u_oracle|: both sides sum nz terms twice, at most
2 nz eps = 4.5e-13 apart."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

TOL = 1e-12


def check(bc, shape, box, precision, zero_mode):
    print(f"singular column {bc} {shape} p{precision} zero_mode={zero_mode}", flush=True)
    f = prng.uniform_pm1(shape, seed=shape[0] + precision)
    ref = oracle.solve(f, bc, box, zero_mode=zero_mode)
    got = pa.solve(f, bc, box, zero_mode=zero_mode, precision=precision)
    err = float(np.abs(got - ref).max() / np.abs(ref).max())
    assert err <= TOL, f"{bc} {shape}: {err:.3e}"
    return f, got


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("nz", [4, 5, 63, 64, 65, 128, 129, 1023, 1024])
def test_singular_column_lengths(nz, precision):
    box = [0, 1, 0, 1, 0, nz / 16.0]
    for bc in ("PPPPPP", "NNNNPP"):
        f, got = check(bc, (nz, 12, 16), box, precision, 1)
        with pa.Batch(precision=precision) as B:
            i = B.add(16, 12, nz, bc, box)
            B.finalize()
            B.set_rhs(i, f)
            B.solve()
            assert np.array_equal(B.get_solution(i), got)
    if precision:
        check("PPPPNN", (nz, 12, 16), box, 1, 1)
        check("NNNNND", (nz, 12, 16), box, 1, 0)

