"""The work a program hands this library, as a list of timed cases.

Every case is one call (or, for a solve or a batch, one whole solve or batch
replay) through the package's public entry points:

  cell     W = A U cell by cell (mass_apply, stiffness_apply, kpm_apply), the
           fused kernels at degrees 1..8 and the high-degree ones at 9..25
  global   y = A x through an int32 dofmap (global_apply)
  affine   the same on affine cells, geometry from 7 values per cell
           (global_apply_affine)
  plan     y = A x through an autotuned Plan on the structured numbering
  batch    an uneven batch of meshes, autotuned, replayed from its graph
  solve    A u = f with PCGSolver to 1e-11

Inputs (tables, dofmaps, geometry, vectors) are made here with torch and numpy
from the seed alone; exact() evaluates the same operators in FP64 with plain
torch tensor contractions.
"""
import math
import random

import numpy as np
import torch

import femtc_amd as F

MASS, STIFF, KPM = F.OP_MASS, F.OP_STIFFNESS, F.OP_KPM
OPS = {"mass": MASS, "stiffness": STIFF, "kpm": KPM}
TYPES = {"f64": torch.float64, "f32": torch.float32}
RTOL = 1e-11


def listed():
    return [
        # Latency: the apply of a very small mesh, as in a coarse level or a
        # unit test; two launches and the call itself.
        {"name": "global_small", "kind": "global", "op": "stiffness",
         "dtype": "f64", "degree": 4, "nq": 5, "nx": 4, "ny": 4, "nz": 4,
         "numbering": "lex"},
        # The cell-local mass apply on 32768 cells: the reference's own
        # bench_mass workload with 5 points per direction.
        {"name": "cell_mass_p3", "kind": "cell", "op": "mass", "dtype": "f64",
         "degree": 3, "nq": 5, "cells": 32768},
        # A cell-local single-precision stiffness apply with over-integration
        # on an odd number of cells.
        {"name": "cell_stiffness_p5_f32", "kind": "cell", "op": "stiffness",
         "dtype": "f32", "degree": 5, "nq": 7, "cells": 20011},
        # High degree: cell-local stiffness at degree 16, about 2e7 dofs.
        {"name": "cell_stiffness_p16", "kind": "cell", "op": "stiffness",
         "dtype": "f64", "degree": 16, "nq": 17, "cells": 4070},
        # The benchmark's apply: stiffness, 48^3 cells, degree 6, any dofmap.
        {"name": "global_stiffness_p6", "kind": "global", "op": "stiffness",
         "dtype": "f64", "degree": 6, "nq": 7, "nx": 48, "ny": 48, "nz": 48,
         "numbering": "lex"},
        # A mesh reader's numbering (dofs in the order the cells first meet
        # them), single precision, odd sizes, over-integrated mass.
        {"name": "global_mass_p3_f32_touch", "kind": "global", "op": "mass",
         "dtype": "f32", "degree": 3, "nq": 5, "nx": 61, "ny": 67, "nz": 71,
         "numbering": "touch"},
        # Affine cells: a Helmholtz-type operator without stored geometry.
        {"name": "affine_kpm_p5", "kind": "affine", "op": "kpm",
         "dtype": "f64", "degree": 5, "nq": 6, "nx": 45, "ny": 46, "nz": 47,
         "numbering": "lex"},
        # Repeated applies of one operator on a structured mesh: a plan, as a
        # time stepper keeps it (64^3 cells, degree 4), and a mass operator.
        {"name": "plan_stiffness_p4", "kind": "plan", "op": "stiffness",
         "dtype": "f64", "degree": 4, "nq": 5, "nx": 64, "ny": 64, "nz": 64},
        {"name": "plan_mass_p7", "kind": "plan", "op": "mass", "dtype": "f64",
         "degree": 7, "nq": 8, "nx": 40, "ny": 41, "nz": 42},
        # Many uneven meshes at once, degrees 2..8, mass and stiffness in
        # turn: the batch benchmark's distribution, fewer and smaller meshes.
        {"name": "batch_uneven", "kind": "batch", "dtype": "f64",
         "meshes": 32, "median_cells": 2000, "spec_seed": 0},
        # The benchmark's solve: (K+M) u = f, FP32 inner iterations with FP64
        # refinement, on the structured grid with affine cells.
        {"name": "solve_refined_p6", "kind": "solve", "op": "kpm",
         "inner": "f32", "affine": True, "degree": 6, "nq": 7, "nx": 48,
         "ny": 48, "nz": 48},
        # A small solve as a request server runs it.
        {"name": "solve_small_p4", "kind": "solve", "op": "kpm",
         "inner": "f32", "affine": True, "degree": 4, "nq": 5, "nx": 8,
         "ny": 8, "nz": 8},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _box(rng, cells):
    """Three cell counts whose product is near `cells`, rarely equal."""
    s = max(1.0, cells) ** (1.0 / 3.0)
    nx = max(1, round(s * rng.uniform(0.75, 1.33)))
    ny = max(1, round(s * rng.uniform(0.75, 1.33)))
    nz = max(1, round(cells / (nx * ny)))
    return nx, ny, nz


def draw(rng: random.Random):
    """One more case: the listed kinds, the whole range of degrees, points,
    types, operators and sizes (over their logarithm)."""
    kind = rng.choice(["cell", "cell_high", "global", "global", "affine",
                       "plan", "plan", "batch", "solve"])
    dtype = rng.choice(["f64", "f64", "f32"])
    op = rng.choice(["mass", "stiffness", "stiffness", "kpm"])
    if kind == "batch":
        return {"kind": "batch", "dtype": dtype,
                "meshes": rng.randint(4, 32),
                "median_cells": int(_log_uniform(rng, 200, 2000)),
                "spec_seed": rng.randrange(1 << 16)}
    if kind == "solve":
        degree = rng.randint(2, 7)
        dofs = _log_uniform(rng, 2e3, 6e6)
        nx, ny, nz = _box(rng, dofs / degree ** 3)
        return {"kind": "solve", "op": rng.choice(["kpm", "kpm", "mass"]),
                "inner": rng.choice(["f32", "f32", "f64"]),
                "affine": rng.random() < 0.7, "degree": degree,
                "nq": degree + rng.choice([1, 1, 2]), "nx": nx, "ny": ny,
                "nz": nz}
    if kind == "cell_high":
        degree = rng.randint(9, 25)
        kind, hi = "cell", 2e7
    else:
        degree, hi = rng.randint(1, 8), 2e7
    nq = degree + rng.choice([1, 1, 2, 3])
    values = _log_uniform(rng, 4e3, hi)
    case = {"kind": kind, "op": op, "dtype": dtype, "degree": degree, "nq": nq}
    if kind == "cell":
        case["cells"] = max(1, int(values / (degree + 1) ** 3))
        return case
    nx, ny, nz = _box(rng, values / degree ** 3)
    case.update(nx=nx, ny=ny, nz=nz)
    if kind != "plan":
        case["numbering"] = rng.choice(["lex", "lex", "touch"])
    return case


# ---- inputs ----------------------------------------------------------------

def _legendre(n, x):
    """P_n and P_n' at x."""
    c = np.zeros(n + 1)
    c[n] = 1.0
    return (np.polynomial.legendre.legval(x, c),
            np.polynomial.legendre.legval(x, np.polynomial.legendre.legder(c)))


def _gll(degree):
    """Gauss-Lobatto-Legendre nodes on [0, 1]."""
    if degree == 1:
        return np.array([0.0, 1.0])
    c = np.zeros(degree + 1)
    c[degree] = 1.0
    x = np.sort(np.real(np.polynomial.legendre.legroots(
        np.polynomial.legendre.legder(c))))
    for _ in range(3):  # Newton on (1 - x^2) P', whose slope is -n(n+1) P
        p, dp = _legendre(degree, x)
        x = x + (1.0 - x * x) * dp / (degree * (degree + 1) * p)
    x = np.concatenate([[-1.0], x, [1.0]])
    return 0.5 * (0.5 * (x - x[::-1]) + 1.0)


def _tables(degree, nq):
    """phi [N][nq], dphi [N][nq] of the GLL Lagrange basis at the Gauss points
    of [0, 1], and the weights."""
    xn = _gll(degree)
    t, w = np.polynomial.legendre.leggauss(nq)
    xq, w = 0.5 * (t + 1.0), 0.5 * w
    n = degree + 1
    phi, dphi = np.ones((n, nq)), np.zeros((n, nq))
    for i in range(n):
        for j in range(n):
            if j != i:
                phi[i] *= (xq - xn[j]) / (xn[i] - xn[j])
        for k in range(n):
            if k == i:
                continue
            term = np.full(nq, 1.0 / (xn[i] - xn[k]))
            for j in range(n):
                if j != i and j != k:
                    term *= (xq - xn[j]) / (xn[i] - xn[j])
            dphi[i] += term
    phi = 0.5 * (phi + phi[::-1, ::-1])
    dphi = 0.5 * (dphi - dphi[::-1, ::-1])
    return phi, dphi, w


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(g, n, dtype):
    return torch.rand(n, generator=g, device="cuda",
                      dtype=torch.float64).mul_(2.0).sub_(1.0).to(dtype)


def _cell_geometry(g, cells):
    """Jacobians J = I + 0.1 U(-1,1) per cell; (J, [cells][7]: |det J| J^-1
    J^-T packed (22, 12, 02, 11, 01, 00), then |det J|), FP64."""
    J = 0.1 * _uniform(g, 9 * cells, torch.float64).view(cells, 3, 3)
    J += torch.eye(3, device="cuda", dtype=torch.float64)
    r0, r1, r2 = J[:, 0], J[:, 1], J[:, 2]
    c0 = torch.linalg.cross(r1, r2)
    c1 = torch.linalg.cross(r2, r0)
    c2 = torch.linalg.cross(r0, r1)
    det = (r0 * c0).sum(1)
    K = torch.stack([c0, c1, c2], dim=2) / det.view(-1, 1, 1)  # J^-1
    a = det.abs()

    def s(i, j):
        return a * (K[:, i] * K[:, j]).sum(1)

    cg = torch.stack([s(2, 2), s(1, 2), s(0, 2), s(1, 1), s(0, 1), s(0, 0), a],
                     dim=1)
    return J.reshape(-1).contiguous(), cg.contiguous()


def _point_geometry(cg, w, nq, dtype, stiffness, mass):
    """G [cells][nq^3][6] and detJw [cells][nq^3] from the per-cell values."""
    w = torch.from_numpy(w).cuda()
    w3 = (w.view(-1, 1, 1) * w.view(1, -1, 1) * w.view(1, 1, -1)).reshape(-1)
    G = D = None
    if stiffness:
        G = torch.empty(cg.shape[0], nq ** 3, 6, device="cuda", dtype=dtype)
        for k in range(6):
            G[:, :, k] = (cg[:, k, None] * w3).to(dtype)
        G = G.view(-1)
    if mass:
        D = (cg[:, 6, None] * w3).to(dtype).reshape(-1)
    return G, D


def _dofmap(nx, ny, nz, degree, numbering):
    """int32 [cells][N^3] and the number of dofs."""
    dev = "cuda"
    P, NY, NZ = degree, ny * degree + 1, nz * degree + 1
    c = torch.arange(nx * ny * nz, device=dev)
    ci, cj, ck = c // (ny * nz), (c // nz) % ny, c % nz
    l = torch.arange((P + 1) ** 3, device=dev)
    a, b, d = l // (P + 1) ** 2, (l // (P + 1)) % (P + 1), l % (P + 1)
    base = (ci * P * NY + cj * P) * NZ + ck * P
    off = (a * NY + b) * NZ + d
    dm = (base[:, None] + off).reshape(-1)
    ndofs = (nx * P + 1) * NY * NZ
    if numbering == "touch":
        first = torch.full((ndofs,), dm.numel(), device=dev)
        first.scatter_reduce_(0, dm, torch.arange(dm.numel(), device=dev),
                              "amin")
        rank = torch.empty_like(first)
        rank[torch.argsort(first)] = torch.arange(ndofs, device=dev)
        dm = rank[dm]
    return dm.to(torch.int32), ndofs


def _mesh_inputs(g, op, dtype, degree, nq, cells, keep_points=True):
    phi, dphi, w = _tables(degree, nq)
    flat = np.concatenate([phi.ravel(), dphi.ravel()])
    J, cg = _cell_geometry(g, cells)
    s = {"tab": torch.from_numpy(flat).to("cuda", dtype), "J": J, "cg": cg,
         "w": w, "G": None, "D": None}
    if keep_points:
        s["G"], s["D"] = _point_geometry(cg, w, nq, dtype, op != MASS,
                                         op != STIFF)
    return s


def _inputs(case, seed):
    """The case's arrays, without any handle of the library."""
    g = _generator(seed)
    op, P, Q = OPS[case["op"]], case["degree"], case["nq"]
    kind = case["kind"]
    if kind == "solve":
        dtype = torch.float64
    else:
        dtype = TYPES[case["dtype"]]
    cells = (case["cells"] if kind == "cell"
             else case["nx"] * case["ny"] * case["nz"])
    keep = kind in ("cell", "global", "plan") or (kind == "solve"
                                                  and not case["affine"])
    s = _mesh_inputs(g, op, dtype, P, Q, cells, keep)
    s.update(op=op, P=P, Q=Q, C=cells, dtype=dtype)
    if kind == "cell":
        n = cells * (P + 1) ** 3
    else:
        s["dm"], n = _dofmap(case["nx"], case["ny"], case["nz"], P,
                             case.get("numbering", "lex"))
    s["n"] = n
    if kind == "affine":
        s["cg"] = s["cg"].to(dtype).reshape(-1)
        s["tabw"] = torch.cat([s["tab"], torch.from_numpy(s["w"]).to("cuda",
                                                                     dtype)])
    s["x"] = _uniform(g, n, dtype)
    return s


def _batch_meshes(case):
    """(degree, operator, box) per mesh: cell counts lognormal about the
    median (sigma 1, clipped to a tenth and ten times it), degrees uniform in
    2..8, operators in turn."""
    rng = random.Random(case["spec_seed"])
    out = []
    for i in range(case["meshes"]):
        m = case["median_cells"]
        cells = min(10 * m, max(m / 10, m * math.exp(rng.gauss(0.0, 1.0))))
        degree = rng.randint(2, 8)
        side = max(1, round(cells ** (1.0 / 3.0)))
        out.append((degree, MASS if i % 2 == 0 else STIFF,
                    (side, side, max(1, math.ceil(cells / side ** 2)))))
    return out


def _batch_items(case, seed):
    g = _generator(seed)
    dtype = TYPES[case["dtype"]]
    items = []
    for degree, op, (nx, ny, nz) in _batch_meshes(case):
        s = _mesh_inputs(g, op, dtype, degree, degree + 1, nx * ny * nz)
        dm, n = _dofmap(nx, ny, nz, degree, "lex")
        items.append({"op": op, "degree": degree, "nq": degree + 1,
                      "tables": s["tab"], "x": _uniform(g, n, dtype),
                      "y": torch.empty(n, device="cuda", dtype=dtype),
                      "G": s["G"], "detJw": s["D"], "dofmap": dm,
                      "num_cells": nx * ny * nz, "ndofs": n,
                      "dims": (nx, ny, nz)})
    return items


def prepare(case, seed):
    if case["kind"] == "batch":
        items = _batch_items(case, seed)
        batch = F.Batch(items)
        batch.autotune(reps=3)
        return {"kind": "batch", "items": items, "batch": batch}
    s = _inputs(case, seed)
    s["kind"] = case["kind"]
    s["y"] = torch.empty(s["n"], device="cuda", dtype=s["dtype"])
    dims = (case.get("nx"), case.get("ny"), case.get("nz"))
    if case["kind"] == "plan":
        s["plan"] = F.Plan(*dims, s["P"], s["dm"], s["n"])
        s["plan"].set_tables(s["tab"], s["Q"])
        s["plan"].autotune(s["op"], None, s["x"], s["y"], s["Q"], G=s["G"],
                           detJw=s["D"], reps=3)
    if case["kind"] == "solve":
        s["solver"] = F.PCGSolver(
            s["op"], s["tab"], s["dm"], s["C"], s["P"], s["Q"], s["n"],
            G=s["G"], detJw=s["D"],
            inner=F.F32 if case["inner"] == "f32" else F.F64,
            J=s["J"] if case["affine"] else None, grid=dims)
    return s


def run(s):
    kind = s["kind"]
    if kind == "batch":
        s["batch"].graph_launch()
        return [it["y"] for it in s["items"]]
    if kind == "cell":
        if s["op"] == MASS:
            F.mass_apply(s["tab"], s["x"], s["y"], s["D"], s["C"], s["P"],
                         s["Q"])
        elif s["op"] == STIFF:
            F.stiffness_apply(s["tab"], s["x"], s["y"], s["G"], s["C"],
                              s["P"], s["Q"])
        else:
            F.kpm_apply(s["tab"], s["x"], s["y"], s["G"], s["D"], s["C"],
                        s["P"], s["Q"])
    elif kind == "global":
        F.global_apply(s["op"], s["tab"], s["x"], s["y"], s["dm"], s["C"],
                       s["P"], s["Q"], G=s["G"], detJw=s["D"])
    elif kind == "affine":
        F.global_apply_affine(s["op"], s["tabw"], s["x"], s["y"], s["dm"],
                              s["C"], s["P"], s["Q"], s["cg"])
    elif kind == "plan":
        s["plan"].apply(s["op"], None, s["x"], s["y"], s["Q"], G=s["G"],
                        detJw=s["D"])
    else:
        s["solver"].solve(s["x"], s["y"], rtol=RTOL)
    return s["y"]


# ---- compulsory work -------------------------------------------------------

def _flops(op, P, Q, cells):
    """Sum-factorised operations: multiply and add counted separately."""
    N = P + 1
    grad, mass = op != MASS, op != STIFF
    one = 2 if grad else 1
    two = 3 if grad else 1
    three = (3 if grad else 0) + (1 if mass else 0)
    line = 2 * (one * N ** 3 * Q + two * N ** 2 * Q ** 2 + three * N * Q ** 3)
    point = (15 if grad else 0) + (1 if mass else 0)
    return cells * (2 * line + point * Q ** 3)


def _apply_work(op, P, Q, cells, dofs, size, dofmap, affine):
    geometry = (0 if op == MASS else 6) + (0 if op == STIFF else 1)
    values = cells * (7 if affine else geometry * Q ** 3)
    moved = size * (2 * dofs + values)
    if dofmap:
        moved += 4 * cells * (P + 1) ** 3
    return {"bytes": moved, "flops": _flops(op, P, Q, cells)}


def work(case):
    """Each array of a call once.  A solve counts its CG iterations: the
    operator, and the passes over the CG vectors that no ordering avoids
    (r, p, e read and written, the diagonal read), 300 iterations being
    typical of the listed solve."""
    kind = case["kind"]
    if kind == "batch":
        total = {"bytes": 0, "flops": 0}
        size = 8 if case["dtype"] == "f64" else 4
        for P, op, (nx, ny, nz) in _batch_meshes(case):
            dofs = (nx * P + 1) * (ny * P + 1) * (nz * P + 1)
            w = _apply_work(op, P, P + 1, nx * ny * nz, dofs, size, True,
                            False)
            total = {k: total[k] + w[k] for k in total}
        return total
    op, P, Q = OPS[case["op"]], case["degree"], case["nq"]
    if kind == "cell":
        return _apply_work(op, P, Q, case["cells"],
                           case["cells"] * (P + 1) ** 3,
                           8 if case["dtype"] == "f64" else 4, False, False)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cells = nx * ny * nz
    dofs = (nx * P + 1) * (ny * P + 1) * (nz * P + 1)
    if kind == "solve":
        size = 8 if case["inner"] == "f64" else 4
        w = _apply_work(op, P, Q, cells, dofs, size, False, case["affine"])
        iters = 300 if op == KPM else 40
        return {"bytes": iters * (w["bytes"] + 7 * size * dofs),
                "flops": iters * (w["flops"] + 12 * dofs)}
    return _apply_work(op, P, Q, cells, dofs,
                       8 if case["dtype"] == "f64" else 4, kind != "plan",
                       kind == "affine")


# ---- the same in 64 bits ---------------------------------------------------

def _along(t, axis, m):
    """Contract axis 1, 2 or 3 of t [cells][..][..][..] with m [in][out]."""
    t = t.movedim(axis, 3).contiguous()
    out = t.reshape(-1, t.shape[3]) @ m
    return out.reshape(*t.shape[:3], m.shape[1]).movedim(3, axis)


def _cell_apply(op, P, Q, tab, U, G, D):
    """W = A U in FP64; U [cells][N][N][N], G [cells][Q][Q][Q][6], D
    [cells][Q][Q][Q] (either may be broadcast over the cells)."""
    N = P + 1
    t = tab.double()
    ph, dp = t[:N * Q].view(N, Q), t[N * Q:2 * N * Q].view(N, Q)
    pT, dT = ph.t().contiguous(), dp.t().contiguous()
    a0, a1 = _along(U, 1, ph), (_along(U, 1, dp) if op != MASS else None)
    b00 = _along(a0, 2, ph)
    W = None
    if op != STIFF:
        v = _along(b00, 3, ph) * D
        W = _along(_along(_along(v, 3, pT), 2, pT), 1, pT)
    if op != MASS:
        d2 = _along(b00, 3, dp)
        d1 = _along(_along(a0, 2, dp), 3, ph)
        d0 = _along(_along(a1, 2, ph), 3, ph)
        g = G
        v0 = g[..., 5] * d0 + g[..., 4] * d1 + g[..., 2] * d2
        v1 = g[..., 4] * d0 + g[..., 3] * d1 + g[..., 1] * d2
        v2 = g[..., 2] * d0 + g[..., 1] * d1 + g[..., 0] * d2
        K = _along(_along(_along(v0, 3, pT), 2, pT), 1, dT)
        K = K + _along(_along(_along(v1, 3, pT), 2, dT)
                       + _along(_along(v2, 3, dT), 2, pT), 1, pT)
        W = K if W is None else W + K
    return W


def _exact_cells(s, U, lo, hi):
    """Cells lo..hi of the operator on the cell values U (FP64)."""
    N, Q, op = s["P"] + 1, s["Q"], s["op"]
    c = hi - lo
    if s["G"] is not None or s["D"] is not None:
        G = D = None
        if op != MASS:
            G = s["G"].view(-1, Q, Q, Q, 6)[lo:hi].double()
        if op != STIFF:
            D = s["D"].view(-1, Q, Q, Q)[lo:hi].double()
    else:
        cg = s["cg"].view(-1, 7)[lo:hi].double()
        w = s.get("w64")
        w3 = w.view(-1, 1, 1) * w.view(1, -1, 1) * w.view(1, 1, -1)
        G = cg[:, None, None, None, :6] * w3[..., None]
        D = cg[:, 6].view(c, 1, 1, 1) * w3
    return _cell_apply(op, s["P"], Q, s["tab"], U.reshape(c, N, N, N), G, D)


def _exact_global(s, x):
    nd = (s["P"] + 1) ** 3
    y = torch.zeros(s["n"], device="cuda", dtype=torch.float64)
    dm = s["dm"].view(s["C"], nd)
    step = max(1, (1 << 26) // max(nd, s["Q"] ** 3))
    for lo in range(0, s["C"], step):
        hi = min(s["C"], lo + step)
        at = dm[lo:hi].reshape(-1).long()
        y.index_add_(0, at, _exact_cells(s, x[at], lo, hi).reshape(-1))
    return y


def _exact_diagonal(s):
    """diag of the continuous operator: the squared and mixed tables."""
    N, Q, op = s["P"] + 1, s["Q"], s["op"]
    t = s["tab"].double()
    ph, dp = t[:N * Q].view(N, Q), t[N * Q:2 * N * Q].view(N, Q)
    m = [(ph * ph).t().contiguous(), (ph * dp).t().contiguous(),
         (dp * dp).t().contiguous()]
    if s["G"] is not None or s["D"] is not None:
        G = s["G"].view(-1, Q, Q, Q, 6) if op != MASS else None
        D = s["D"].view(-1, Q, Q, Q) if op != STIFF else None
    else:
        w = s["w64"]
        w3 = w.view(-1, 1, 1) * w.view(1, -1, 1) * w.view(1, 1, -1)
        cg = s["cg"].view(-1, 7)
        G = cg[:, None, None, None, :6] * w3[..., None]
        D = cg[:, 6].view(-1, 1, 1, 1) * w3
    d = 0
    if op != STIFF:
        d = _along(_along(_along(D, 1, m[0]), 2, m[0]), 3, m[0])
    if op != MASS:
        for k, f, (i, j, l) in ((5, 1, (2, 0, 0)), (3, 1, (0, 2, 0)),
                                (0, 1, (0, 0, 2)), (4, 2, (1, 1, 0)),
                                (2, 2, (1, 0, 1)), (1, 2, (0, 1, 1))):
            d = d + f * _along(_along(_along(G[..., k], 1, m[i]), 2, m[j]), 3,
                               m[l])
    y = torch.zeros(s["n"], device="cuda", dtype=torch.float64)
    return y.index_add_(0, s["dm"].long(), d.reshape(-1))


def _exact_solve(s):
    """Jacobi-PCG in FP64 to 1e-13."""
    inv = 1.0 / _exact_diagonal(s)
    u = torch.zeros_like(s["x"])
    r = s["x"].clone()
    z = inv * r
    p = z.clone()
    rz, stop = torch.dot(r, z), 1e-13 * float(r.norm())
    for it in range(5000):
        ap = _exact_global(s, p)
        alpha = rz / torch.dot(p, ap)
        u += alpha * p
        r -= alpha * ap
        if it % 8 == 7 and float(r.norm()) <= stop:
            break
        z = inv * r
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
    return u


def exact(case, seed):
    if case["kind"] == "batch":
        out = []
        for it in _batch_items(case, seed):
            s = {"op": it["op"], "P": it["degree"], "Q": it["nq"],
                 "tab": it["tables"], "G": it["G"], "D": it["detJw"],
                 "dm": it["dofmap"], "C": it["num_cells"], "n": it["ndofs"]}
            out.append(_exact_global(s, it["x"].double()))
        return out
    s = _inputs(case, seed)
    s["w64"] = torch.from_numpy(s["w"]).cuda()
    if case["kind"] == "affine":
        s["w64"] = s["tabw"][2 * (s["P"] + 1) * s["Q"]:].double()
    if case["kind"] == "cell":
        U = s["x"].double()
        nd = (s["P"] + 1) ** 3
        out = torch.empty(s["n"], device="cuda", dtype=torch.float64)
        step = max(1, (1 << 26) // max(nd, s["Q"] ** 3))
        for lo in range(0, s["C"], step):
            hi = min(s["C"], lo + step)
            out[lo * nd:hi * nd] = _exact_cells(s, U[lo * nd:hi * nd], lo,
                                                hi).reshape(-1)
        return out
    if case["kind"] == "solve":
        return _exact_solve(s)
    return _exact_global(s, s["x"].double())
