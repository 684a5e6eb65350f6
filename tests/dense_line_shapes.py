"""Grids whose lines of up to 128 points without a compiled plan run as dense products of lines (the other
axis is too long for the plane kernel), and one row fewer where that is a matter of their number:
(shape (nz, ny, nx), boundary conditions, axis, is the axis dense).  tests/test_dispatch_rules.py holds them
against the rules, so that a later rule cannot send them elsewhere unseen."""
KINDS = ["DD", "NN", "PP", "ND", "DN"]  # numbered as the library's
LENGTHS = [2, 3, 5, 13, 15, 17, 31, 33, 34, 63, 65, 94, 127]


def shapes(kind, n):
    quarter = kind in ("ND", "DN")
    # (the oracle, like the reference, takes periodic x with periodic y only)
    x_bc = kind + ("PPDD" if kind == "PP" else "NNDD")
    few = n <= 112  # any number of folded lines; quarter-wave lines along x from 2048
    out = []
    if quarter or not few:
        out += [((16, 128, n), x_bc, 0, True), ((23, 89, n), x_bc, 0, False)]
    else:
        out += [((5, 70, n), x_bc, 0, True), ((4, 67, n), x_bc, 0, True)]
    if quarter and not few:
        out += [((16, n, 128), "NN" + kind + "DN", 1, True), ((23, n, 89), "DD" + kind + "DD", 1, False)]
    else:
        out += [((5, n, 70), "NN" + kind + "DN", 1, True), ((4, n, 67), "DD" + kind + "DD", 1, True)]
    # (two points are the convolution's)
    return [(s, bc, axis, dense and n > 2) for s, bc, axis, dense in out]
