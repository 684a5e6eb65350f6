"""The serving form's matrices of long dense-product lines: they take no device memory beside the pool,
however many lengths a server meets; in a pool far smaller than the matrices of all its requests they
give way to each other; and a request whose region fits the pool only without them runs as convolutions.

Bars: results bitwise the single solves, where a request keeps its matrices; else max-norm difference
<= 1e-12 relative to max|u_oracle|, the FP64 bar of every parity test.  Device memory: resident tables of
the lengths met, below 0.5 MB each (two lengths' matrices alone are 13 MB)."""
import numpy as np
import pytest

import oracle
import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

LONG = list(range(701, 1001, 13))


def test_device_memory_stays_in_the_pool():
    import torch

    with pa.Server(hbm_bytes=1 << 30, staging_bytes=1 << 20, streams=2) as S:
        S.wait(S.submit((48, 701, 64), "DDNNDD", want_solution=False))
        before = torch.cuda.mem_get_info()[0]
        for n in LONG:
            print(f"server length {n}", flush=True)
            S.wait(S.submit((48, n, 64), "NNNNDD", seed=n, want_solution=False))
        grown = before - torch.cuda.mem_get_info()[0]
        assert grown <= len(LONG) * (1 << 19), f"{grown / 1e6:.1f} MB beside the pool"


@pytest.mark.parametrize("precision", [0, 1])
def test_matrices_give_way_in_a_small_pool(precision):
    # y lines of 67 .. 199 points (matrices of up to 0.33 MB, 8 MB all together), x and z lines between
    shapes = [(10 + i % 5, n, 17 + i % 3) for i, n in enumerate(range(67, 200, 4))]
    shapes += [(9, 33, n) for n in range(69, 110, 6)] + [(n, 18, 20) for n in (71, 73, 97)]
    kinds = ["NNNNDD", "DDDDNN", "NNPPDD", "DDDNDN", "NNNDDD"]
    cases = [(s, "NNNNPP" if s[0] > 64 else kinds[i % 5]) for i, s in enumerate(shapes)]
    with pa.Server(hbm_bytes=4 << 20, staging_bytes=64 << 20, streams=3) as S:
        rhs = [prng.uniform_pm1(s, seed=i) for i, (s, _) in enumerate(cases)]
        for again in range(2):
            tickets = [S.submit(s, bc, precision=precision, rhs=f) for (s, bc), f in zip(cases, rhs)]
            for t, (s, bc), f in zip(tickets, cases, rhs):
                print(f"small pool {bc} {s} precision={precision}", flush=True)
                assert np.array_equal(S.wait(t)[0], pa.solve(f, bc, precision=precision)), (s, bc)


@pytest.mark.parametrize("shape,bc", [((9, 101, 16), "NNNNDD"), ((9, 16, 101), "DDNNDD"), ((101, 12, 14), "NNNNPP")])
def test_no_room_for_matrices(shape, bc):
    print(f"no room {bc} {shape}", flush=True)
    f = prng.uniform_pm1(shape, seed=3)
    ref = oracle.solve(f, bc, zero_mode=1)
    with pa.Server(hbm_bytes=64 << 20, staging_bytes=1 << 20, streams=1) as S:
        room = S.footprint(shape, bc)
    # one unit of the pool less than region and matrices: accepted as convolutions, in less room
    with pa.Server(hbm_bytes=room - 256, staging_bytes=1 << 20, streams=1) as S:
        less = S.footprint(shape, bc)
        assert less < room - 256
        got = S.wait(S.submit(shape, bc, rhs=f))[0]
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
    # exactly enough for both, after another request's matrices lay in the way
    with pa.Server(hbm_bytes=room, staging_bytes=1 << 20, streams=1) as S:
        other = (4, 67, 9)
        S.wait(S.submit(other, "NNDDDD", rhs=prng.uniform_pm1(other, seed=1)))
        got = S.wait(S.submit(shape, bc, rhs=f))[0]
        assert S.footprint(shape, bc) == room
    assert np.array_equal(got, pa.solve(f, bc))
