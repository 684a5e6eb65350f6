"""Performance cases of the solve path: what a program that uses this library has it do.

A case is one call pattern on one problem size, through the package's public classes:

  solve   PoissonHIP on device arrays (the flow-solver pattern: the right-hand side and the
          solution stay in HBM, one solve per time step), FP64 or mixed precision, optionally
          replayed from a HIP graph;
  host    PoissonHIP in the reference's own call order on host arrays: assignRhs, pittPack,
          getSolution;
  batch   Batch: many small grids of different sizes and boundary conditions in one call;
  serve   Server: independent requests of any size from host arrays, solutions to host arrays.

Boxes have nearly cubic cells, right-hand sides are uniform in [-1, 1].  `exact` solves the same
cell-centred 7-point system by dense eigenvector products in FP64.
"""
import math
import random

import numpy as np
import torch

import pittpack_amd as pa

XY_KINDS = ("PP", "NN", "DD", "ND", "DN")
Z_KINDS = ("DD", "NN", "DN", "ND", "PP")
# sides of the batched workload's grids in x and y (z: any length from 16 to 256)
BATCH_SIDES = (32, 48, 64, 96, 128, 192)


def listed():
    return [
        # the smallest grid a program solves in a loop: latency and launches are all it costs
        {"name": "tiny_24x20x18", "kind": "solve", "nx": 24, "ny": 20, "nz": 18, "bc": "NNDDDN", "precision": 0, "graph": 0,
         "stretch": 1.0},
        # a channel in a time loop: periodic in x and y, walls in z, replayed from a captured graph
        {"name": "cube_64_graph", "kind": "solve", "nx": 64, "ny": 64, "nz": 64, "bc": "PPPPNN", "precision": 0,
         "graph": 1, "stretch": 1.0},
        # the reference's main program: host arrays in and out, its boundary conditions
        {"name": "host_128", "kind": "host", "nx": 128, "ny": 128, "nz": 128, "bc": "NNNNDD", "precision": 0, "graph": 0,
         "stretch": 1.0},
        # a cavity on a medium grid whose planes are small
        {"name": "box_128x96x320", "kind": "solve", "nx": 128, "ny": 96, "nz": 320, "bc": "DDNNDN", "precision": 0,
         "graph": 0, "stretch": 1.0},
        # homogeneous turbulence: periodic in all three directions
        {"name": "cube_256_periodic", "kind": "solve", "nx": 256, "ny": 256, "nz": 256, "bc": "PPPPPP", "precision": 0,
         "graph": 0, "stretch": 1.0},
        # the largest: a half-channel with long lines and columns, quarter-wave in y, stretched cells
        {"name": "half_channel_1024x768x640", "kind": "solve", "nx": 1024, "ny": 768, "nz": 640, "bc": "PPNDNN",
         "precision": 0, "graph": 0, "stretch": 1.2},
        # sides nobody rounded: odd and prime
        {"name": "odd_101x97x89", "kind": "solve", "nx": 101, "ny": 97, "nz": 89, "bc": "DDNNDD", "precision": 0,
         "graph": 0, "stretch": 1.0},
        # a larger grid of such sides
        {"name": "odd_331x202x277", "kind": "solve", "nx": 331, "ny": 202, "nz": 277, "bc": "NNPPDD", "precision": 0,
         "graph": 0, "stretch": 0.9},
        # the benchmark grid, FP64 and in the mixed-precision form
        {"name": "cube_512", "kind": "solve", "nx": 512, "ny": 512, "nz": 512, "bc": "DDNDDD", "precision": 0,
         "graph": 0, "stretch": 1.0},
        {"name": "mixed_512x512x256", "kind": "solve", "nx": 512, "ny": 512, "nz": 256, "bc": "DDNDDD", "precision": 1,
         "graph": 0, "stretch": 1.0},
        # many small grids at once
        {"name": "batch_48", "kind": "batch", "members": 48, "mix": 2, "precision": 0},
        # requests of any size, FP64 and mixed, host to host
        {"name": "serve_16", "kind": "serve", "requests": 16, "mix": 5, "lo": 32, "hi": 160},
    ]


def draw(rng):
    kind = rng.choice(["solve"] * 7 + ["host", "batch", "serve"])
    if kind == "batch":
        return {"kind": "batch", "members": rng.randint(8, 48), "mix": rng.randrange(1 << 30),
                "precision": int(rng.random() < 0.3)}
    if kind == "serve":
        return {"kind": "serve", "requests": rng.randint(4, 16), "mix": rng.randrange(1 << 30), "lo": 32, "hi": 160}

    def side(lo, hi):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        # half of all programs round their grids
        return n if rng.random() < 0.5 else max(lo, (n + 15) // 16 * 16)

    hi, most = (1024, 1 << 27) if kind == "solve" else (192, 1 << 23)
    n = [side(16, hi) for _ in range(3)]
    while n[0] * n[1] * n[2] > most:
        n = [side(16, hi) for _ in range(3)]
    return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2],
            "bc": rng.choice(XY_KINDS) + rng.choice(XY_KINDS) + rng.choice(Z_KINDS),
            "precision": int(kind == "solve" and rng.random() < 0.2), "graph": int(kind == "solve" and rng.random() < 0.3),
            "stretch": round(rng.uniform(0.8, 1.25), 3)}


def _box(nx, ny, nz, stretch):
    """near-cubic cells: dx = dz, dy = stretch * dz, the longest side of length about 1"""
    h = 1.0 / max(nx, ny, nz)
    return [0.0, nx * h, 0.0, ny * h * stretch, 0.0, nz * h]


def _problems(case):
    """the case's grids: (nx, ny, nz, bc, box, precision) each"""
    if case["kind"] in ("solve", "host"):
        n = (case["nx"], case["ny"], case["nz"])
        return [n + (case["bc"], _box(*n, case["stretch"]), case["precision"])]
    r = random.Random(case["mix"])
    out = []
    if case["kind"] == "batch":
        for _ in range(case["members"]):
            n = (r.choice(BATCH_SIDES), r.choice(BATCH_SIDES), r.randint(16, 256))
            bc = r.choice(("PPPP", "PPNN", "NNPP", "NNNN", "DDDD", "DDNN")) + r.choice(("DD", "NN"))
            out.append(n + (bc, _box(*n, 1.0), case["precision"]))
        return out
    for _ in range(case["requests"]):
        n = tuple(int(round(math.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]))))) for _ in range(3))
        bc = r.choice(("PPPP", "PPNN", "NNPP", "NNNN", "DDDD")) + r.choice(("DD", "NN"))
        out.append(n + (bc, _box(*n, 1.0), r.randrange(2)))
    return out


def _rhs(nx, ny, nz, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    f = torch.rand((nz, ny, nx), generator=g, device="cuda", dtype=torch.float64)
    return f.mul_(2.0).sub_(1.0)


_solver_stream = None


def _stream():
    """the one stream this program solves on (graph replay needs a stream of its own)"""
    global _solver_stream
    if _solver_stream is None:
        _solver_stream = torch.cuda.Stream()
    return _solver_stream.cuda_stream


class _DeviceArray:
    """a device pointer of the library as an array torch can view"""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "data": (ptr, False), "version": 3,
                                         "strides": None}


def prepare(case, seed):
    probs = _problems(case)
    kind = case["kind"]
    if kind in ("solve", "host"):
        nx, ny, nz, bc, box, prec = probs[0]
        M = pa.PoissonHIP(nx, ny, nz)
        M.assignBoundary(bc)
        M.setBox(box)
        M.setCoords(2)
        if prec:
            M.set_option(pa.OPT_PRECISION, prec)
        if kind == "host":
            return {"kind": kind, "M": M, "f": _rhs(nx, ny, nz, seed).cpu().numpy()}
        M.set_stream(_stream())
        if case["graph"]:
            M.set_option(pa.OPT_GRAPH, 1)
        f = _rhs(nx, ny, nz, seed)
        u = torch.empty_like(f)
        torch.cuda.synchronize()
        return {"kind": kind, "M": M, "f": f, "u": u}
    if kind == "batch":
        B = pa.Batch(precision=case["precision"])
        for nx, ny, nz, bc, box, _ in probs:
            B.add(nx, ny, nz, bc, box)
        B.finalize()
        B.set_stream(_stream())
        shapes = [(nz, ny, nx) for nx, ny, nz, _, _, _ in probs]
        for i, s in enumerate(shapes):
            torch.as_tensor(_DeviceArray(B.field_ptr(i), s, B), device="cuda").copy_(_rhs(s[2], s[1], s[0], seed * 64 + i))
        u = [torch.as_tensor(_DeviceArray(B.solution_ptr(i), s, B), device="cuda") for i, s in enumerate(shapes)]
        torch.cuda.synchronize()
        return {"kind": kind, "B": B, "u": u}
    S = pa.Server(hbm_bytes=4 << 30, staging_bytes=1 << 29, streams=4)
    f = [_rhs(p[0], p[1], p[2], seed * 64 + i).cpu().numpy() for i, p in enumerate(probs)]
    return {"kind": kind, "S": S, "f": f, "probs": probs}


def run(state):
    kind = state["kind"]
    if kind == "solve":
        state["M"].solve_device_oop(state["f"].data_ptr(), state["u"].data_ptr())
        return state["u"]
    if kind == "host":
        M = state["M"]
        M.assignRhs(state["f"])
        M.pittPack()
        return M.getSolution()
    if kind == "batch":
        state["B"].solve()
        return state["u"]
    S = state["S"]
    tickets = [S.submit((p[2], p[1], p[0]), p[3], box=p[4], precision=p[5], rhs=f)
               for p, f in zip(state["probs"], state["f"])]
    return [S.wait(t)[0] for t in tickets]


def work(case):
    nbytes = flops = 0.0
    for nx, ny, nz, _, _, _ in _problems(case):
        pts = float(nx) * ny * nz
        nbytes += 16.0 * pts  # the right-hand side in, the solution out
        # forward and inverse real transforms in x and y, two sweeps in z
        flops += pts * (2 * 2.5 * (math.log2(nx) + math.log2(ny)) + 8.0)
    return {"bytes": nbytes, "flops": flops}


# ---- the same system in plain torch, FP64 ----------------------------------------------------


def _basis(n, kind, dev):
    """orthonormal eigenvectors (columns) and eigenvalues of the 1D cell-centred second difference"""
    j = torch.arange(n, device=dev, dtype=torch.float64)[:, None]
    k = torch.arange(n, device=dev, dtype=torch.float64)[None, :]
    if kind == "PP":
        m = torch.div(k + 1, 2, rounding_mode="floor")  # constant, then cosine and sine of 1, 2, ...
        ang = torch.remainder(j * m, n) * (2 * math.pi / n)
        q = torch.where((torch.remainder(k, 2) == 1) | (k == 0), torch.cos(ang), torch.sin(ang))
        theta = m[0] * (2 * math.pi / n)
    else:
        # angles as whole multiples of pi / (4 n), reduced before they are evaluated
        num = {"NN": 4 * k, "DD": 4 * (k + 1), "ND": 4 * k + 2, "DN": 4 * k + 2}[kind]  # theta = num pi / (4 n)
        ang = torch.remainder(num * (2 * j + 1) / 2, 8 * n) * (math.pi / (4 * n))
        q = torch.cos(ang) if kind in ("NN", "ND") else torch.sin(ang)
        theta = num[0] * (math.pi / (4 * n))
    q = q / torch.linalg.vector_norm(q, dim=0, keepdim=True)
    return q, -4.0 * torch.sin(theta / 2) ** 2


def _face_value(omega, x, tag):
    return math.cos(omega * x) if tag == 1 else 0.0 if tag == 2 else math.sin(omega * x)


def _effective_rhs(f, bc, box):
    """f dz^2 minus the boundary data of the Dirichlet faces (the library's built-in face values)"""
    nz, ny, nx = f.shape
    n = (nx, ny, nz)
    h = [(box[2 * a + 1] - box[2 * a]) / n[a] for a in range(3)]
    tags = []
    for a in range(3):
        p = bc[2 * a:2 * a + 2]
        tags.append({"DD": 0, "NN": 1, "PP": 2}.get(p, -1))
    if bc[4] in "DN":
        tags[2] = -1 if bc[4] == "D" else -2
    elif "ND" not in (bc[:2], bc[2:4]) and "DN" not in (bc[:2], bc[2:4]):
        tags[2] = -1  # no other direction is the untransformed one
    om = [math.pi, 2 * math.pi, 3 * math.pi]
    e = [torch.tensor([_face_value(om[a], box[2 * a] + (i + 0.5) * h[a], tags[a]) for i in range(n[a])],
                      device=f.device, dtype=torch.float64) for a in range(3)]
    face = [[_face_value(om[a], box[2 * a + s], tags[a]) for s in range(2)] for a in range(3)]
    g = f * (h[2] * h[2])
    for s, at in ((0, 0), (1, -1)):
        if bc[0 + s] == "D":
            g[:, :, at] -= 2 * face[0][s] * e[2][:, None] * e[1][None, :]
        if bc[2 + s] == "D":
            g[:, at, :] -= 2 * face[1][s] * e[2][:, None] * e[0][None, :]
        if bc[4 + s] == "D":
            g[at] -= 2 * face[2][s] * e[1][:, None] * e[0][None, :]
    return g, (h[2] / h[0]) ** 2, (h[2] / h[1]) ** 2


def _singular_column(r, periodic):
    """the z column of the constant x-y mode where the operator is singular: its first row is
    replaced by u_0 = r_0, or by u_0 + u_{n-1} = (r_0 + r_{n-1}) / 2 where z is periodic"""
    r = r.astype(np.longdouble)
    n = len(r)
    if not periodic:
        d = -np.cumsum(r[::-1])[::-1]  # d_i = u_i - u_{i-1}
        return np.concatenate([r[:1], r[0] + np.cumsum(d[1:])]).astype(np.float64)
    R = np.concatenate([[np.longdouble(0)], np.cumsum(r[1:n - 1])])  # d_{i+1} = d_1 + R_i
    d1 = -(r[n - 1] + R.sum() + R[n - 2]) / n
    s = np.concatenate([[np.longdouble(0)], np.cumsum(d1 + R)])
    return ((r[0] + r[n - 1]) / 4 - s[-1] / 2 + s).astype(np.float64)


def _solve_exact(f, bc, box):
    nz, ny, nx = f.shape
    g, Cx, Cy = _effective_rhs(f, bc, box)
    qx, lx = _basis(nx, bc[0:2], f.device)
    qy, ly = _basis(ny, bc[2:4], f.device)
    qz, lz = _basis(nz, bc[4:6], f.device)
    g = torch.matmul(g.reshape(-1, nx), qx).reshape(nz, ny, nx)
    g = torch.matmul(qy.t().contiguous(), g)
    singular = all(k in ("PP", "NN") for k in (bc[0:2], bc[2:4], bc[4:6]))
    if singular:
        column = _singular_column(g[:, 0, 0].cpu().numpy(), bc[4] == "P")
    g = torch.matmul(qz.t().contiguous(), g.reshape(nz, -1)).reshape(nz, ny, nx)
    for k in range(nz):
        lam = Cx * lx[None, :] + Cy * ly[:, None] + lz[k]
        if singular and k == 0:
            lam[0, 0] = 1.0
        g[k] /= lam
    g = torch.matmul(qz, g.reshape(nz, -1)).reshape(nz, ny, nx)
    if singular:
        g[:, 0, 0] = torch.from_numpy(column).to(f.device)
    g = torch.matmul(qy, g)
    return torch.matmul(g.reshape(-1, nx), qx.t().contiguous()).reshape(nz, ny, nx)


def exact(case, seed):
    out = []
    for i, (nx, ny, nz, bc, box, _) in enumerate(_problems(case)):
        one = case["kind"] in ("solve", "host")
        u = _solve_exact(_rhs(nx, ny, nz, seed if one else seed * 64 + i), bc, box)
        out.append(u.cpu().numpy() if case["kind"] in ("host", "serve") else u)
    return out[0] if case["kind"] in ("solve", "host") else out
