"""Cell-local applies at nq = 6, whose workgroups pack 7 cells over 4 waves
from 4096 cells (mass) and 32768 cells (FP32 stiffness and K+M) on: the last
count before each, every remainder by 7 behind it, against the oracle cell by
cell; nothing is written past the output.  The cells repeat 41 different ones,
so a cell that takes another's data shows.

Bars as for the other cell-local applies: 1e-12 (FP64), 1e-5 (FP32)."""
import numpy as np
import pytest

import femtc_amd as F
import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = {torch.float64: 1e-12, torch.float32: 1e-5}


@pytest.mark.parametrize("P", [3, 4, 5])
@pytest.mark.parametrize("dt", [torch.float64, torch.float32],
                         ids=["f64", "f32"])
@pytest.mark.parametrize("op", ["mass", "stiffness", "kpm"])
def test_packed_cells_vs_oracle(op, dt, P):
    Q, N = 6, P + 1
    nl, some = N ** 3, 41
    tab = O.basis_tables(P, Q)
    U = O.uniform(P, some * nl)
    G = O.uniform(P + 1, some * Q ** 3 * 6, 0.0, 1.0)
    Dw = O.uniform(P + 2, some * Q ** 3, 0.5, 1.5)
    ref = O.cell_operator(op, N, Q, tab, U, G, Dw, some).reshape(some, nl)
    least = 4096 if op == "mass" else 32768
    most = least + 7

    def many(a):
        t = torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dt)
        return t.repeat((most + some - 1) // some)

    dtab = torch.from_numpy(tab).to("cuda", dt)
    dU, dG, dD = many(U), many(G), many(Dw)
    dref = torch.from_numpy(ref).to("cuda").repeat((most + some - 1) // some,
                                                   1)
    for C in (1, 7, 50, least - 1, *range(least, most)):
        print(f"packed {op} {dt} P={P} cells={C}", flush=True)
        W = torch.full((C * nl + 64,), -5.0, device="cuda", dtype=dt)
        out = W[:C * nl]
        if op == "mass":
            F.mass_apply(dtab, dU[:C * nl], out, dD[:C * Q ** 3], C, P, Q)
        elif op == "stiffness":
            F.stiffness_apply(dtab, dU[:C * nl], out, dG[:C * Q ** 3 * 6], C,
                              P, Q)
        else:
            F.kpm_apply(dtab, dU[:C * nl], out, dG[:C * Q ** 3 * 6],
                        dD[:C * Q ** 3], C, P, Q)
        torch.cuda.synchronize()
        assert (W[C * nl:] == -5.0).all()
        d = (out.double().view(C, nl) - dref[:C]).norm(dim=1)
        assert (d / dref[:C].norm(dim=1)).max().item() <= TOL[dt]
