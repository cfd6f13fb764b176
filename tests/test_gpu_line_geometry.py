"""The line kernels' two ways to the geometry (staged through LDS, or read by
the line with several points in flight) against the general kernel on the GPU:
the smallest shapes of either, a last chunk that is not full, a last pass over
a few lines only, and two-cell workgroups that run half a cell apart, with as
few cells as bring them there and a last cell without a partner.

Bars: the two kernels round the same products and differ in the order of
their sums, at most 6 contractions of 28 terms: 168 roundings of 1.1e-16 (FP64)
and 6.0e-8 (FP32) are 1.9e-14 and 1.0e-5 in the worst case without
cancellation, and add up at random to a tenth of it; the suite's 1e-12 and 1e-5
hold the rest.
"""
import pytest

import femtc_amd as F
import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = {torch.float64: 1e-12, torch.float32: 1e-5}


def _pairs_apart():
    # four pairs of cells per CU: from there on a workgroup of two staged
    # cells takes several pairs
    return 8 * torch.cuda.get_device_properties(0).multi_processor_count


SHAPES = [
    (9, 10, 37, False), (11, 12, 37, False), (11, 13, 37, False),
    (11, 14, 37, False), (13, 14, 41, False), (13, 16, 41, False),
    (15, 16, 1029, False), (21, 22, 13, False), (23, 24, 13, False),
    (25, 26, 5, False),
    (16, 17, -3, True), (16, 17, -1, True), (16, 17, 3, True),
    (15, 18, 1, True), (17, 18, 2, True), (20, 21, 1, True),
]


@pytest.mark.parametrize("P,Q,ncell,apart", SHAPES)
@pytest.mark.parametrize("dt", [torch.float64, torch.float32],
                         ids=["f64", "f32"])
@pytest.mark.parametrize("op", ["mass", "stiffness", "kpm"])
def test_line_geometry_vs_general(op, dt, P, Q, ncell, apart):
    if apart:
        ncell += _pairs_apart()
    print(f"line geometry {op} {dt} P={P} Q={Q} cells={ncell}", flush=True)
    nl = (P + 1) ** 3
    gen = torch.Generator(device="cuda").manual_seed(17 * P + Q)

    def rand(n, lo, hi, off=0):
        t = torch.empty(n + off, device="cuda", dtype=dt)
        t.uniform_(lo, hi, generator=gen)
        return t[off:]

    tab = torch.from_numpy(O.basis_tables(P, Q)).to("cuda", dt)
    U = rand(ncell * nl, -1.0, 1.0)
    G = rand(ncell * Q ** 3 * 6, 0.0, 1.0)
    # one value past a pair's alignment, which detJw need not have
    D = rand(ncell * Q ** 3, 0.5, 1.5, 1)
    out = {}
    for mode in (F.HIGH_DEGREE_AUTO, F.HIGH_DEGREE_GENERAL):
        W = torch.full((ncell * nl + 64,), -7.0, device="cuda", dtype=dt)
        Wc = W[:ncell * nl]
        with F.high_degree_kernel(mode):
            if op == "mass":
                F.mass_apply(tab, U, Wc, D, ncell, P, Q)
            elif op == "stiffness":
                F.stiffness_apply(tab, U, Wc, G, ncell, P, Q)
            else:
                F.kpm_apply(tab, U, Wc, G, D, ncell, P, Q)
        torch.cuda.synchronize()
        assert (W[ncell * nl:] == -7.0).all()
        out[mode] = Wc.double()
    a, b = out[F.HIGH_DEGREE_AUTO], out[F.HIGH_DEGREE_GENERAL]
    # every cell by itself: one wrong cell of thousands would not show in the
    # norm over all of them
    d = (a - b).view(ncell, nl).norm(dim=1) / b.view(ncell, nl).norm(dim=1)
    assert d.max().item() <= TOL[dt], (op, P, Q, int(d.argmax()))
