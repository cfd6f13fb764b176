"""The chain kernel behind the one-shot gathered applies: every kind of
numbering it must merge or must not merge faces for, chains that end short,
cells straddling waves (Q = 6), overwrite and accumulate, against the oracle,
on boxes of more cells than its count (FROM); the same numberings on a few
cells, which the atomic kernel runs.

The kernel sums the same products as the atomic scatter in another order, so
the bars are those of the gathered applies: 1e-12 (FP64), 1e-5 (FP32)."""
import numpy as np
import pytest

import femtc_amd as F
import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = {torch.float64: 1e-12, torch.float32: 1e-5}


def numbered(kind, dims, P, seed=1):
    """(dofmap, number of dofs) of the box `dims`, in the numbering `kind`."""
    nx, ny, nz = dims
    nd = (P + 1) ** 3
    dm = O.dofmap_structured(nx, ny, nz, P).reshape(-1, nd)
    ng = (nx * P + 1) * (ny * P + 1) * (nz * P + 1)
    rng = np.random.default_rng(seed)
    if kind == "reader":  # dofs in the order the cells first meet them
        _, first = np.unique(dm, return_index=True)
        rank = np.empty(ng, dtype=np.int64)
        rank[np.argsort(first)] = np.arange(ng)
        dm = rank[dm]
    elif kind == "relabelled":
        dm = rng.permutation(ng)[dm]
    elif kind == "shuffled":  # consecutive cells share a face by chance only
        dm = dm[rng.permutation(len(dm))]
    elif kind == "periodic":  # the last cell of a z-line closes on its first
        last = dm.reshape(nx, ny, nz, P + 1, P + 1, P + 1)
        last[:, :, -1, :, :, -1] = last[:, :, 0, :, :, 0]
    elif kind == "partial":  # one edge of each face is not shared
        for k in range(1, len(dm)):
            cell = dm[k].reshape(P + 1, P + 1, P + 1)
            cell[0, :, 0] = cell[0, ::-1, 0].copy()
    return np.ascontiguousarray(dm.ravel(), dtype=np.int32), ng


def check(op, P, Q, dims, kind, dtype, affine=False, accumulate=False):
    N, C = P + 1, int(np.prod(dims))
    dm, ng = numbered(kind, dims, P)
    J = O.random_jacobians(5, C)
    G, Dw = O.geometry_affine(J, Q)
    tab = O.basis_tables(P, Q)
    x = O.uniform(11, ng)
    y0 = O.uniform(12, ng)
    ref = O.global_operator(op, N, Q, tab, x, dm, G, Dw)
    if accumulate:
        ref = ref + y0

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)

    y = dev(y0)
    code = {"mass": F.OP_MASS, "stiffness": F.OP_STIFFNESS,
            "kpm": F.OP_KPM}[op]
    ddm = torch.from_numpy(dm).cuda()
    if affine:
        cg = torch.empty(C * 7, device="cuda", dtype=dtype)
        F.geometry_cell(torch.from_numpy(J).cuda(), cg)
        F.global_apply_affine(code, dev(F.basis_tables_weights(P, Q)), dev(x),
                              y, ddm, C, P, Q, cg, accumulate=accumulate)
    else:
        F.global_apply(code, dev(tab), dev(x), y, ddm, C, P, Q, G=dev(G),
                       detJw=dev(Dw), accumulate=accumulate)
    torch.cuda.synchronize()
    got = y.double().cpu().numpy()
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= TOL[dtype], (op, P, Q, dims, kind, dtype, err)


KINDS = ["lex", "reader", "relabelled", "shuffled", "periodic", "partial"]
# chains of 32, 14, 8, 7 (cells over the 4 waves at Q = 6), 4 and 3 cells:
# lines shorter than, equal to and longer than a chain
SHAPES = [(1, 2, (2, 2, 9)), (2, 3, (2, 3, 5)), (3, 5, (2, 2, 7)),
          (4, 5, (1, 3, 8)), (5, 6, (2, 2, 5)), (3, 6, (1, 2, 4)),
          (6, 7, (1, 2, 5)), (7, 8, (1, 2, 4))]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("P,Q,dims", SHAPES)
def test_numberings(P, Q, dims, kind):
    for op in ("mass", "stiffness", "kpm"):
        for dtype in (torch.float64, torch.float32):
            check(op, P, Q, dims, kind, dtype)
            check(op, P, Q, dims, kind, dtype, affine=True, accumulate=True)


@pytest.mark.parametrize("P,Q", [(P, Q) for P in range(1, 9)
                                 for Q in range(P + 1, min(P + 4, 10))])
def test_chain_ends(P, Q):
    """One cell, and counts around the chain's length."""
    for nz in (1, 2, 3, 7, 8, 15, 33):
        check("mass", P, Q, (1, 1, nz), "lex", torch.float64,
              accumulate=nz % 2 == 1)
        check("kpm", P, Q, (1, 1, nz), "reader", torch.float32, affine=True)


def test_periodic_single_cell():
    """A cell whose own right and left faces are the same dofs."""
    for P, Q in ((1, 2), (4, 5), (5, 6), (7, 8)):
        check("mass", P, Q, (2, 2, 1), "periodic", torch.float64)
        check("stiffness", P, Q, (2, 2, 1), "periodic", torch.float32,
              affine=True)


@pytest.mark.parametrize("kind", ["lex", "reader", "relabelled"])
@pytest.mark.parametrize("P", [1, 2, 3, 4])
def test_plan_that_was_not_tuned(P, kind):
    """A plan's first apply: direct but for degree 1 FP64 stiffness, K+M."""
    Q, dims = P + 1, (3, 5, 17)
    dm, ng = numbered(kind, dims, P)
    C = int(np.prod(dims))
    G, Dw = O.geometry_affine(O.random_jacobians(5, C), Q)
    tab, x = O.basis_tables(P, Q), O.uniform(11, ng)
    y0 = O.uniform(12, ng)
    plan = F.Plan(*dims, P, torch.from_numpy(dm).cuda(), ng)
    for op, code in (("mass", F.OP_MASS), ("stiffness", F.OP_STIFFNESS),
                     ("kpm", F.OP_KPM)):
        ref = O.global_operator(op, P + 1, Q, tab, x, dm, G, Dw)
        for dtype, dt in ((torch.float64, F.F64), (torch.float32, F.F32)):
            blocked = P == 1 and dt == F.F64 and op != "mass"
            assert plan.get_block(Q, dt, code) == ((1, 2, 16) if blocked
                                                   else (0, 0, 0))
            dtab, dx, dG, dD, y = (torch.from_numpy(a).to("cuda", dtype)
                                   for a in (tab, x, G, Dw, y0))
            for accumulate in (False, True):
                plan.apply(code, dtab, dx, y, Q, G=dG, detJw=dD,
                           accumulate=accumulate)
            torch.cuda.synchronize()
            got = y.double().cpu().numpy()
            err = np.linalg.norm(got - 2 * ref) / np.linalg.norm(2 * ref)
            assert err <= TOL[dtype], (op, P, kind, dtype, err)


# cells from which the chain kernel runs at (P, Q) (FP64 and FP32)
FROM = {(1, 2): 10240, (1, 3): 24576, (1, 4): 8192, (2, 3): 6144,
        (2, 4): 6144, (2, 5): 6144, (3, 4): 2048, (3, 5): 5120, (3, 6): 5120,
        (4, 5): 3072, (4, 6): 4096, (4, 7): 4096, (5, 6): 2048, (5, 7): 3072,
        (5, 8): 3072, (6, 7): 1280, (6, 8): 1280, (7, 8): 1280}
CODE = {"mass": F.OP_MASS, "stiffness": F.OP_STIFFNESS, "kpm": F.OP_KPM}


def compare(P, Q, dm, ng, ops, accumulate=False):
    """Gathered applies of every op, both types, per-point and affine geometry,
    against the oracle."""
    N = P + 1
    C = len(dm) // N ** 3
    J = O.random_jacobians(5, C)
    G, Dw = O.geometry_affine(J, Q)
    tab, x, y0 = O.basis_tables(P, Q), O.uniform(11, ng), O.uniform(12, ng)
    ddm = torch.from_numpy(dm).cuda()
    for op in ops:
        ref = O.global_operator(op, N, Q, tab, x, dm, G, Dw)
        if accumulate:
            ref = ref + y0
        for dtype in (torch.float64, torch.float32):
            def dev(a):
                return torch.from_numpy(np.ascontiguousarray(a)).to("cuda",
                                                                    dtype)
            cg = torch.empty(C * 7, device="cuda", dtype=dtype)
            F.geometry_cell(torch.from_numpy(J).cuda(), cg)
            for affine in (False, True):
                y = dev(y0)
                if affine:
                    F.global_apply_affine(
                        CODE[op], dev(F.basis_tables_weights(P, Q)), dev(x), y,
                        ddm, C, P, Q, cg, accumulate=accumulate)
                else:
                    F.global_apply(CODE[op], dev(tab), dev(x), y, ddm, C, P, Q,
                                   G=dev(G), detJw=dev(Dw),
                                   accumulate=accumulate)
                torch.cuda.synchronize()
                got = y.double().cpu().numpy()
                err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
                assert err <= TOL[dtype], (op, P, Q, dtype, affine, err)


# z-lines shorter than, equal to and longer than a chain, as in SHAPES
BOXES = [(1, 2, (25, 46, 9)), (2, 3, (31, 40, 5)), (3, 5, (27, 28, 7)),
         (4, 5, (13, 30, 8)), (5, 6, (19, 22, 5)), (3, 6, (32, 41, 4)),
         (6, 7, (13, 20, 5)), (7, 8, (18, 18, 4)), (4, 7, (4, 30, 35)),
         (1, 3, (24, 32, 33))]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("P,Q,dims", BOXES)
def test_numberings_from_the_count(P, Q, dims, kind):
    assert np.prod(dims) >= FROM[P, Q]
    compare(P, Q, *numbered(kind, dims, P), ("mass", "stiffness", "kpm"),
            accumulate=kind in ("reader", "shuffled"))


@pytest.mark.parametrize("P,Q", sorted(FROM))
def test_chain_ends_from_the_count(P, Q):
    """Last chains of one to three cells, and just short of full."""
    for more in (1, 3, 31):
        compare(P, Q, *numbered("lex", (1, 1, FROM[P, Q] + more), P),
                ("mass",))


def operator_kernels(call):
    """Names of the operator kernels that call() launches."""
    from torch.profiler import ProfilerActivity, profile

    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return {e.key for e in prof.key_averages()
            if "apply_cells<" in e.key or "chain_cells<" in e.key}


@pytest.mark.parametrize("P,Q", sorted(FROM))
def test_kernel_by_count(P, Q):
    """The atomic kernel below the count, the chain kernel from it on."""
    N = P + 1
    for dtype in (torch.float64, torch.float32):
        at = 0 if (P, Q, dtype) == (1, 4, torch.float32) else FROM[P, Q]
        for C in (max(at - 1, 1), max(at, 1)):
            dm = torch.arange(C * N ** 3, device="cuda", dtype=torch.int32)
            x = torch.ones(C * N ** 3, device="cuda", dtype=dtype)
            y = torch.empty_like(x)
            D = torch.ones(C * Q ** 3, device="cuda", dtype=dtype)
            tab = torch.from_numpy(O.basis_tables(P, Q)).to("cuda", dtype)
            ran = operator_kernels(lambda: F.global_apply(
                F.OP_MASS, tab, x, y, dm, C, P, Q, detJw=D))
            assert len(ran) == 1, ran
            assert ("chain_cells" in ran.pop()) == (C >= at), (P, Q, C)


def chained_in_part(P, nz, rows, links, seed=3):
    """(dofmap, number of dofs) of `rows` rows of nz cells along z, where cell
    k (k > 0) of a row shares its left face with cell k-1 only if k is in
    `links`; dofs in random order."""
    N = P + 1
    row = np.empty((nz, N, N, N), dtype=np.int64)
    n = 0
    for k in range(nz):
        first = 0
        if k in links:
            row[k, :, :, 0] = row[k - 1, :, :, P]
            first = 1
        new = N * N * (N - first)
        row[k, :, :, first:] = n + np.arange(new).reshape(N, N, N - first)
        n += new
    dm = row[None] + n * np.arange(rows)[:, None, None, None, None]
    dm = np.random.default_rng(seed).permutation(n * rows)[dm]
    return np.ascontiguousarray(dm.ravel(), dtype=np.int32), n * rows


# the kernel looks at the first two pairs of a chain: merged cells where it
# takes the whole chain for unmerged, and single cells where it merges, at every
# place of a chain (rows of 9 and 34 cells; P=5: cells straddling waves)
LINKS = [set(), {1}, {2}, {3, 4, 6}, {1, 5}, {2, 4, 6, 8}, {1, 2, 3},
         set(range(1, 40))]


@pytest.mark.parametrize("P,Q", [(1, 2), (2, 3), (4, 5), (5, 6), (6, 7),
                                 (7, 8)])
@pytest.mark.parametrize("links", LINKS)
def test_chained_in_part(P, Q, links):
    for nz in (9, 34):
        rows = -(-FROM[P, Q] // nz)
        compare(P, Q, *chained_in_part(P, nz, rows, links), ("mass", "kpm"))


def test_no_loss_where_nothing_chains():
    """FP32 mass P=7 on cells whose local axes are rotated, so that the cells
    after one another share their a-faces and the dofs run along a: as many
    atomics as dofs of the cells, but no more than 3 times the time of the
    numbering that chains (5 times when every cell was written in runs along
    c; 1.4 when its lanes write it)."""
    P, Q, n = 7, 8, 20
    N, C = P + 1, n ** 3
    dm, ng = numbered("lex", (n, n, n), P)
    rot = np.ascontiguousarray(
        dm.reshape(C, N, N, N).transpose(0, 3, 1, 2).ravel())
    tab = torch.from_numpy(O.basis_tables(P, Q)).to("cuda", torch.float32)
    D = torch.rand(C * Q ** 3, device="cuda")
    x = torch.rand(ng, device="cuda")
    y = torch.empty_like(x)
    ms = []
    for m in (dm, rot):
        m = torch.from_numpy(m).cuda()
        best = 1e9
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(10):
                F.global_apply(F.OP_MASS, tab, x, y, m, C, P, Q, detJw=D)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        ms.append(best)
    assert ms[1] <= 3 * ms[0], ms
