"""A batch's captured solve runs a stage's shape classes as branches of one graph: every replay, with
new right-hand sides and eager work of the program between them, bitwise the batch launched one by one.
Classes from one to many, small planes, dense lines, long, periodic and singular columns, both forms."""
import numpy as np
import pytest
import torch

import pittpack_amd as pa
from pittpack_amd import rng as prng

pytestmark = pytest.mark.gpu

BIG = (256, 256, 160, "NNDDDD")  # past the 10 million points from which there are branches
ONE = [BIG, (256, 256, 155, "NNDDDD")]
MANY = [(16, 24, 18, "NNDDDD"), (24, 16, 18, "DDNNNN"), (48, 48, 64, "PPPPNN"), (64, 32, 40, "NNPPDD"), (96, 48, 100, "DDDDDD"),
        (31, 33, 16, "NDDNDD"), (70, 66, 21, "NNNNNN"), (32, 32, 48, "PPPPPP"), (24, 24, 45, "PPPPPP"), (48, 16, 600, "NNNNDD"),
        (64, 64, 64, "NNNNNN"), BIG]


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("members", [ONE, MANY], ids=["one", "many"])
def test_replays_are_the_eager_solve(members, precision):
    if precision:
        members = [m for m in members if m[2] <= 512]
    print(f"batch branches {len(members)} members precision={precision}", flush=True)
    batches = []
    for graph in (0, 1):
        B = pa.Batch(precision=precision)
        B.set_option(pa.OPT_GRAPH, graph)
        for nx, ny, nz, bc in members:
            B.add(nx, ny, nz, bc, [0, 1, 0, 1, 0, 1])
        B.finalize()
        batches.append(B)
    busy = torch.ones(1 << 20, device="cuda")
    for replay in range(5):
        for B in batches:
            for i, (nx, ny, nz, _) in enumerate(members):
                B.set_rhs(i, prng.uniform_pm1((nz, ny, nx), seed=100 * replay + i))
            B.solve()
            busy.mul_(1.5).sum().item()
        for i in range(len(members)):
            eager, got = (B.get_solution(i) for B in batches)
            assert np.array_equal(eager, got), f"replay {replay} member {i} {members[i]}"
    for B in batches:
        B.close()
