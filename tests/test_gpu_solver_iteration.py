"""The CG iteration's fused scalar steps at the sizes where they change: one
block, one value per thread, the most blocks, and energies summed by the
update itself or combined first; and a solve that breaks down (p.Ap not
positive) ends with an error on every block and leaves the solver usable.

Solutions are checked by their residual, re-evaluated by the oracle, at the
solve's own tolerance plus the rounding of the operator (1e-12)."""
import numpy as np
import pytest

import femtc_amd as F
import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def problem(dims, P, G=None):
    nx, ny, nz = dims
    C, Q = nx * ny * nz, P + 1
    ng = (nx * P + 1) * (ny * P + 1) * (nz * P + 1)
    J = O.random_jacobians(3, C)
    g, Dw = O.geometry_affine(J, Q)
    return {"P": P, "Q": Q, "C": C, "ng": ng, "tab": O.basis_tables(P, Q),
            "dm": O.dofmap_structured(nx, ny, nz, P), "dims": dims,
            "G": g if G is None else G(g), "D": Dw}


def solver(p, inner, scatter):
    dev = {k: torch.from_numpy(np.ascontiguousarray(p[k])).cuda()
           for k in ("tab", "dm", "G", "D")}
    return F.PCGSolver(F.OP_KPM, dev["tab"], dev["dm"], p["C"], p["P"],
                       p["Q"], p["ng"], G=dev["G"], detJw=dev["D"],
                       inner=inner, grid=p["dims"], scatter=scatter)


# 27, 125 and 4913 dofs (1, 1 and 20 blocks); 5202 one-cell waves (energies
# combined first) on 97,675 dofs; 274,625 dofs (1024 blocks, several values
# per thread)
@pytest.mark.parametrize("dims,P", [((1, 1, 1), 2), ((2, 2, 2), 2),
                                    ((4, 4, 4), 4), ((17, 17, 18), 5),
                                    ((32, 32, 32), 2)])
@pytest.mark.parametrize("inner", [F.F64, F.F32])
@pytest.mark.parametrize("scatter", [F.SCATTER_DIRECT, F.SCATTER_ASSEMBLED,
                                     F.SCATTER_ZRUN])
def test_sizes(dims, P, inner, scatter):
    p = problem(dims, P)
    f = O.uniform(7, p["ng"])
    u = torch.empty(p["ng"], device="cuda", dtype=torch.float64)
    with solver(p, inner, scatter) as S:
        for _ in range(2):
            info = S.solve(torch.from_numpy(f).cuda(), u, rtol=1e-10)
    uh = u.cpu().numpy()
    r = f - O.global_operator("kpm", P + 1, p["Q"], p["tab"], uh, p["dm"],
                              p["G"], p["D"])
    assert np.linalg.norm(r) / np.linalg.norm(f) <= 1.0e-10 + 1e-12, info


@pytest.mark.parametrize("inner", [F.F64, F.F32])
@pytest.mark.parametrize("scatter", [F.SCATTER_DIRECT, F.SCATTER_ASSEMBLED])
def test_breakdown(inner, scatter):
    """Geometry with an off-diagonal entry over its diagonal ones: the
    operator is indefinite (p.Ap < 0 at the fourth step), its diagonal not."""
    def indefinite(g):
        g = g.reshape(-1, 6).copy()
        g[:, 4] = 1.2 * g[:, 5]
        return g.ravel()

    p = problem((6, 6, 6), 3, indefinite)
    f = torch.from_numpy(O.uniform(7, p["ng"])).cuda()
    u = torch.empty(p["ng"], device="cuda", dtype=torch.float64)
    with solver(p, inner, scatter) as S:
        for _ in range(2):
            info = S.solve(f, u, rtol=1e-10, maxit=500, check=False)
            assert info["status"] == F._lib.ERR_BREAKDOWN, info


def operator_kernels(call):
    """Names of the operator kernels that call() launches."""
    from torch.profiler import ProfilerActivity, profile

    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return {e.key for e in prof.key_averages()
            if "apply_cells<" in e.key or "chain_cells<" in e.key}


@pytest.mark.parametrize("inner", [F.F64, F.F32])
@pytest.mark.parametrize("structured", [True, False])
def test_timed_operators_are_the_solves(inner, structured):
    """The scatters and forms tried at creation are timed on the kernels that
    a CG iteration launches (which write the energies of p.Ap): not on the
    chain kernel, which has none (and runs applies of this many cells), and
    the chosen one among them."""
    p = problem((13, 13, 13), 3)
    if not structured:
        p["dims"] = None
    made = []
    tried = operator_kernels(
        lambda: made.append(solver(p, inner, F.SCATTER_AUTO)))
    assert tried and not any("chain_cells" in k for k in tried), tried
    f = torch.from_numpy(O.uniform(7, p["ng"])).cuda()
    u = torch.empty_like(f)
    with made[0] as S:
        S.set_batch(4, False)
        run = operator_kernels(lambda: S.solve(f, u, rtol=1e-10))
    # (a refined solve's FP64 residual has kernels of its own)
    name = "apply_cells<" + ("double" if inner == F.F64 else "float")
    run = {k for k in run if name in k}
    assert run and run <= tried, (run, tried)
