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
    # four pairs of cells per CU: workgroups of two staged cells (from three
    # pairs per CU on) take several pairs
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


# (P, Q, cells per CU, cells more): either side of the counts from which a
# shape is staged -- 3 pairs per CU for two cells of a workgroup, half and a
# quarter of a cell per CU for FP32 stiffness and K+M of one -- and the smallest
# staged shapes with their neighbours by the line
EDGES = [
    (16, 17, 6, -2), (16, 17, 6, -1), (16, 17, 6, 1), (14, 17, 6, 1),
    (17, 20, 6, -3), (17, 20, 6, 0), (21, 22, 0.5, -1), (21, 22, 0.5, 0),
    (22, 23, 0.25, -1), (22, 23, 0.25, 0), (11, 14, 0.5, -1),
    (11, 14, 0.5, 1), (11, 14, 0, 1), (12, 14, 0, 37), (12, 15, 0, 37),
    (15, 17, 0, 1029), (15, 18, 0, 37), (17, 18, 0, 37), (21, 24, 0, 13),
]


@pytest.mark.parametrize("P,Q,per_cu,more", EDGES)
@pytest.mark.parametrize("dt", [torch.float64, torch.float32],
                         ids=["f64", "f32"])
@pytest.mark.parametrize("op", ["stiffness", "kpm"])
def test_line_geometry_edges(op, dt, P, Q, per_cu, more):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    test_line_geometry_vs_general(op, dt, P, Q, int(per_cu * cus) + more,
                                  False)


def test_few_pairs_per_cu():
    """FP32 K+M at P=16, Q=19 (two cells of 6 waves each) takes about as long
    per cell with 2 pairs of cells per CU as with 8: 1.2 times, and 1.5 times
    when the pairs were staged in step."""
    P, Q = 16, 19
    N = P + 1
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    tab = torch.from_numpy(O.basis_tables(P, Q)).to("cuda", torch.float32)
    per_cell = []
    for C in (4 * cus - 8, 16 * cus):
        U = torch.rand(C * N ** 3, device="cuda")
        W = torch.empty_like(U)
        G = torch.rand(C * Q ** 3 * 6, device="cuda")
        D = torch.rand(C * Q ** 3, device="cuda")
        best = 1e9
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                F.kpm_apply(tab, U, W, G, D, C, P, Q)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        per_cell.append(best / C)
    assert per_cell[0] <= 1.35 * per_cell[1], per_cell
