"""Host rules that choose a transform's kernel, compiled for the host alone (tests/dispatch_rules.cpp): the
table layout of the no-allocation entry point, the y blocks that z tiles rest on,
the routes that the tests of short dense lines mean to take, and on which side of the rules the grids lie whose
two routes have been measured."""
import ctypes
import os
import random
import subprocess

import pytest

import dense_line_shapes

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    from pittpack_amd import build

    so = str(tmp_path_factory.mktemp("rules") / "librules.so")
    subprocess.run([build.hipcc(), "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-fPIC",
                    "-shared", "-I" + build.SRC, "-I" + os.path.join(ROOT, "include"),
                    os.path.join(HERE, "dispatch_rules.cpp"), "-o", so], check=True, capture_output=True)
    L = ctypes.CDLL(so)
    L.rule_dense.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long]
    L.rule_dense_waves.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long]
    L.rule_dense_waves.restype = ctypes.c_long
    L.rule_y_block.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long]
    return L


def layout(rules, nx, ny, nz, bc, one_pass):
    starts, ends = (ctypes.c_long * 32)(), (ctypes.c_long * 32)()
    count, room = ctypes.c_int(0), ctypes.c_long(0)
    bits = rules.rule_noalloc(nx, ny, nz, bc.encode(), int(one_pass), starts, ends, ctypes.byref(count), ctypes.byref(room))
    return bits, sorted(zip(starts[: count.value], ends[: count.value])), room.value


def test_noalloc_axes_keep_the_matrices_that_fit(rules):
    """one axis whose matrices do not fit does not cost the others theirs"""
    for shape, bc, axes in (((101, 509, 97), "DDNNDD", 1), ((509, 101, 97), "NNDDDD", 2), ((101, 97, 331), "NNNNPP", 3 | 4),
                            ((331, 331, 331), "PPPPPP", 1 | 2 | 4), ((401, 1021, 8), "NNNNDD", 1), ((24, 20, 18), "NNDDDD", 3),
                            ((64, 64, 701), "NNNNPP", 4), ((64, 64, 767), "NNNNPP", 0)):
        bits = layout(rules, *shape, bc, False)[0]
        assert bits & 8 and bits & 7 == axes, (shape, bc, bits & 7)


def test_noalloc_layouts_fit_and_do_not_overlap(rules):
    rng = random.Random(7)
    kinds = ["PP", "NN", "DD", "ND", "DN"]
    sizes = [2, 3, 4, 17, 33, 63, 64, 65, 101, 331, 439, 509, 620, 701, 1021, 1023, 1024]
    for _ in range(4000):
        n = [rng.choice(sizes) if rng.random() < 0.6 else rng.randint(2, 1024) for _ in range(3)]
        bc = "".join(rng.choice(kinds) for _ in range(3))
        for one_pass in (False, True) if bc.endswith("PP") else (False,):
            bits, spans, room = layout(rules, *n, bc, one_pass)
            assert bits & 8, (n, bc)
            assert spans[0][0] >= 0 and spans[-1][1] <= room, (n, bc)
            assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:])), (n, bc, spans)
            assert all(a % 32 == 0 for a, _ in spans)


def test_y_blocks_divide_a_z_tile(rules):
    """every FP64 y launch's columns fill a 16-column z tile in whole blocks"""
    for n in range(2, 1025):
        for kind in range(5):
            for nx, lines in ((4, 16), (500, 100000)):
                cols = rules.rule_y_block(n, kind, nx, lines)
                assert cols > 0 and 16 % cols == 0, (n, kind, nx, lines, cols)


@pytest.mark.parametrize("kind", dense_line_shapes.KINDS)
def test_short_dense_line_shapes_take_their_route(rules, kind):
    number = {k: i for i, k in enumerate(dense_line_shapes.KINDS)}
    lanes = set()
    for n in dense_line_shapes.LENGTHS:
        for (nz, ny, nx), bc, axis, dense in dense_line_shapes.shapes(kind, n):
            kx, ky = number[bc[:2]], number[bc[2:4]]
            lines = (nx if axis else ny) * nz
            got = not rules.rule_plane(nx, ny, kx, ky) and bool(rules.rule_dense(n, (kx, ky)[axis], axis, nx, lines))
            assert got == dense, (n, (nz, ny, nx), bc, axis)
            if axis == 0 and dense:
                lanes.add(rules.rule_stage_lanes(n, kx))
    assert lanes == {8, 16, 32, 64}


DD, NN, PP, ND, DN = range(5)
# (n, kind, axis, other two extents) -> time of a solve with dense lines / with convolutions, on an MI355X
MEASURED = [
    # y lines in few columns, which the products pad to 16
    ((331, NN, 1, 4, 960), 1.14), ((509, NN, 1, 4, 960), 1.52), ((1021, PP, 1, 4, 960), 2.32), ((254, NN, 1, 4, 960), 0.92),
    ((1021, NN, 1, 12, 320), 1.43), ((401, NN, 1, 12, 320), 0.86), ((1021, PP, 1, 40, 128), 1.18), ((767, PP, 1, 40, 128), 0.83),
    ((767, NN, 1, 8, 512), 1.03), ((613, NN, 1, 8, 512), 0.85), ((767, NN, 1, 4, 960), 1.69), ((1021, NN, 1, 128, 128), 0.90),
    ((201, ND, 1, 4, 960), 1.15), ((331, DN, 1, 4, 960), 1.60), ((130, ND, 1, 4, 960), 0.87), ((94, ND, 1, 4, 960), 0.63),
    ((127, ND, 1, 4, 960), 0.70), ((331, ND, 1, 12, 320), 1.03), ((509, ND, 1, 12, 320), 1.44), ((254, DN, 1, 12, 320), 0.87),
    ((401, ND, 1, 40, 128), 1.07), ((331, ND, 1, 40, 128), 0.89), ((254, ND, 1, 8, 512), 1.11), ((509, ND, 1, 128, 128), 0.86),
    ((250, ND, 1, 20, 160), 1.10), ((193, ND, 1, 8, 296), 1.03), ((254, ND, 1, 20, 200), 0.87), ((201, ND, 1, 96, 44), 0.85),
    # quarter-wave x lines
    ((201, ND, 0, 96, 22), 1.10), ((254, ND, 0, 96, 24), 1.16), ((255, DN, 0, 128, 32), 1.05), ((254, ND, 0, 512, 128), 1.05),
    ((185, DN, 0, 96, 32), 1.07), ((279, ND, 0, 96, 32), 1.05), ((201, ND, 0, 128, 64), 0.93), ((222, ND, 0, 128, 128), 0.96),
    ((138, ND, 0, 96, 22), 0.97), ((271, ND, 0, 128, 64), 0.75), ((254, NN, 0, 96, 32), 0.98),
    # units in rounds of 256
    ((767, NN, 1, 96, 44), 0.89), ((1021, NN, 1, 96, 44), 1.30), ((1021, PP, 1, 96, 64), 1.05), ((1021, NN, 1, 96, 42), 0.90),
    ((897, NN, 1, 96, 53), 1.10), ((897, NN, 1, 96, 74), 0.87), ((613, NN, 1, 96, 44), 0.75), ((509, NN, 1, 96, 44), 0.84),
    ((331, ND, 1, 96, 44), 0.88), ((401, DN, 1, 96, 44), 1.06), ((509, ND, 1, 96, 64), 1.08), ((509, ND, 1, 96, 85), 0.94),
    ((371, NN, 0, 96, 44), 1.07), ((371, NN, 0, 96, 64), 0.93), ((439, PP, 0, 96, 48), 1.14), ((439, NN, 0, 96, 74), 0.92),
    ((613, NN, 0, 96, 44), 1.24), ((613, DD, 0, 96, 85), 0.84), ((523, NN, 0, 96, 44), 1.08), ((331, NN, 0, 96, 53), 0.93),
    ((185, ND, 0, 96, 44), 1.10), ((185, ND, 0, 96, 85), 0.90), ((213, DN, 0, 96, 88), 1.05), ((280, ND, 0, 96, 44), 1.03),
    ((280, ND, 0, 96, 64), 0.89), ((155, ND, 0, 96, 64), 0.91),
    # very short lines
    ((2, NN, 0, 128, 32), 1.04), ((2, PP, 1, 512, 512), 1.55), ((3, ND, 1, 512, 512), 1.31), ((4, NN, 0, 512, 512), 1.07),
    ((5, NN, 1, 128, 128), 0.97), ((7, NN, 1, 512, 512), 1.22), ((13, ND, 1, 512, 512), 1.15), ((15, PP, 1, 512, 128), 1.06),
    ((13, NN, 0, 512, 512), 0.80), ((17, NN, 1, 512, 512), 0.93), ((3, NN, 1, 96, 8), 0.97), ((7, PP, 0, 96, 24), 0.93),
]


def test_the_faster_route(rules):
    for (n, kind, axis, a, b), ratio in MEASURED:
        cols, lines = (a, a * b) if axis else (n, a * b)
        assert bool(rules.rule_dense(n, kind, axis, cols, lines)) == (ratio < 1), (n, kind, axis, a, b, ratio)


def test_short_dense_lines_bring_waves(rules):
    """at least a wave a unit (with half of that, 1024 units of short lines and 1056 of quarter-wave ones were
    slower than the convolution)"""
    for n in list(range(2, 65)) + [65, 94, 127, 170, 201]:
        for kind in range(5):
            for axis in (0, 1):
                for units in (64, 256, 512, 1024, 1056):
                    assert rules.rule_dense_waves(n, kind, axis, units) >= units, (n, kind, axis, units)


def test_fused_correction_shapes(rules):
    """elements a thread holds of a line in the fused correction step, as measured: eight of 64 and 128 points
    (four: up to 1.6 times slower), half of what the narrow shape has of 32 and 80"""
    assert [rules.rule_resx_elements(n) for n in (32, 64, 80, 128, 256, 512)] == [4, 8, 10, 8, 8, 8]


def test_periodic_z_blocks_are_whole_waves_on_all_banks(rules):
    slots = ctypes.c_int(0)
    served = [nz for nz in range(8, 1025, 2) if rules.rule_zper(nz, ctypes.byref(slots))]
    assert len(served) == 29 and served[:4] == [8, 10, 12, 14]
    for nz in served:
        assert rules.rule_zper(nz, ctypes.byref(slots)) % 64 == 0, nz
        # 16 columns' first elements on the 64 banks, four banks each
        assert len({4 * slots.value * col % 64 for col in range(16)}) == 16, (nz, slots.value)
