"""Shapes on both sides of the lines where the rules choose another form of
the line solve: how many workgroups share a CU, and whether all lines run at
once.

Non-periodic lines: every form of a family rounds alike, so the solution is
bit for bit that of a form pinned by its variant (plain: six-row ring; twisted:
the same).  Periodic lines: against the reference's order on the same factors
in complex double (a few units of rounding a row: 1e-12), complex float against
complex double (records carry 6e-8 each: 1e-5)."""
import pytest

pytestmark = pytest.mark.gpu


def _lines(torch, L, n, seed, periodic=False):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    mat = torch.randn((L * n, 5, 5, 5), dtype=torch.complex128, generator=g, device="cuda") * 0.14
    for k in range(5):
        mat[:, k, k, 2] += 3.0
    rhs = torch.randn((L * n, 5), dtype=torch.complex128, generator=g, device="cuda")
    if periodic:                      # layout 2: the last row of a line repeats the first
        rhs.reshape(L, n, 5)[:, -1] = rhs.reshape(L, n, 5)[:, 0]
    return mat, rhs


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


PLAIN = [(0, L, n) for L, n in ((1025, 157), (1025, 158), (1025, 162), (1537, 158), (1541, 172), (1541, 173))] + \
        [(1, L, n) for L, n in ((600, 59), (600, 60), (1025, 163), (1025, 164), (1540, 84), (1600, 158), (2049, 163), (2050, 164))]
TWISTED = [(0, 513, 311), (0, 513, 312), (0, 769, 129), (0, 769, 160), (0, 1025, 129), (1, 513, 323), (1, 769, 200), (1, 1024, 163), (1, 1025, 322),
           (1, 1025, 324)]


@pytest.mark.parametrize("prec,L,n,twisted", [c + (0,) for c in PLAIN] + [c + (1,) for c in TWISTED])
def test_forms_by_the_rule(prec, L, n, twisted):
    from lns3d_amd.native import Penta, set_line_variant
    torch = _torch()
    print(f"form by the rule L={L} n={n} prec={prec} twisted={twisted}", flush=True)
    layout = 1 + n % 2
    mat, rhs = _lines(torch, L, n, L + n)
    got = []
    try:
        for variant in ((2, 5) if twisted else (0, 3)):
            set_line_variant(n, L, prec, variant)
            h = Penta(0, layout, L, n, prec)
            h.factor(mat)
            x = rhs.clone()
            h.solve(x)
            torch.cuda.synchronize()
            got.append(x)
            h.close()
    finally:
        set_line_variant(n, L, prec, -1)
    assert torch.equal(torch.view_as_real(got[0]).view(torch.int64), torch.view_as_real(got[1]).view(torch.int64))
    assert bool(torch.isfinite(got[0].abs()).all())


# rows stored; unknowns are one fewer.  (513, 87), (513, 257) and the like: the
# last row count of a form and the first of the next
PERIODIC = [(513, 87), (513, 88), (513, 257), (515, 258), (512, 48), (512, 49), (3, 294), (3, 295), (3, 638), (3, 639),
            (513, 126), (515, 127), (514, 294), (513, 295)]


@pytest.mark.parametrize("L,n", PERIODIC)
def test_periodic_forms_by_the_rule(L, n):
    from lns3d_amd.native import Penta
    torch = _torch()
    print(f"periodic form by the rule L={L} n={n}", flush=True)
    mat, rhs = _lines(torch, L, n, L + n, periodic=True)
    h, h32 = Penta(1, 2, L, n, 0, exact=1), Penta(1, 2, L, n, 1, exact=1)
    h.factor(mat)
    h32.factor(mat)
    want, x, x32 = rhs.clone(), rhs.clone(), rhs.clone()
    h.solve_reference_order(want)
    h.solve(x)
    h32.solve(x32)
    torch.cuda.synchronize()
    scale = float(want.abs().max())
    assert float((x - want).abs().max()) < 1e-12 * scale
    assert float((x32 - want).abs().max()) < 1e-5 * scale
    h.close()
    h32.close()
