"""The streaming line solve (line_solve.hpp) at the edges of its forms: lines
of fewer rows than a chunk, of whole chunks and one row more or less, both
families, an odd line count in plain pairs, and the shapes where the form
changes (resident right-hand sides or a ring, three-, six- and twelve-row
chunks).  Against the oracle's cpenta_bc.

Tolerances: the lines are diagonally dominant, so a solve's error is a few
units of rounding per row, well below 1e-12 in complex double; complex-float
records carry 6e-8 each, 1e-5 over the lines' effective coupling length."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


# (lines, rows, variant or None): every row count around a chunk, then the
# shapes at which the form changes
EDGES = [(1, n, None) for n in (7, 8, 11, 12, 13, 16, 17, 18, 23, 24, 25, 26, 29, 30, 31, 36, 37, 47, 48, 49, 50)]
PLAIN = [(3, n, v) for n in (7, 12, 15, 16, 27, 28, 36) for v in (0, 1, 3, 4)]
TWISTED = [(2, n, v) for n in (16, 17, 27, 28, 40, 41) for v in (2, 5, 6)]
SHAPES = [(2, 1400, None), (257, 340, None), (513, 16, None), (513, 165, 2), (769, 40, None), (1025, 19, 2),
          (515, 330, 2), (1027, 200, None)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("lines,n,variant", EDGES + PLAIN + TWISTED + SHAPES)
def test_line_forms(torch_cuda, orc, lines, n, variant, prec):
    from lns3d_amd.native import Penta, set_line_variant
    from tests.penta_cases import random_lines, relerr
    torch = torch_cuda
    layout = 1 + n % 2
    print(f"line form lines={lines} n={n} variant={variant} prec={prec}", flush=True)
    mat, rhs = random_lines(lines, n, layout, seed=7 * lines + n)
    m_ref, x_ref = mat.copy(order="F"), rhs.copy(order="F")
    orc.cpenta_bc(layout, m_ref, x_ref, 2)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.reshape(-1, order="F"))).to("cuda")
    try:
        if variant is not None:
            set_line_variant(n, lines, prec, variant)
        h = Penta(0, layout, lines, n, prec)
        dm, dr = dev(mat), dev(rhs)
        h.factor(dm)
        for _ in range(2):          # a second solve finds the LDS as the first left it
            dr.copy_(dev(rhs))
            h.solve(dr)
        assert relerr(dr.cpu().numpy().reshape(rhs.shape, order="F"), x_ref) < (1e-12 if prec == 0 else 1e-5)
        h.close()
    finally:
        if variant is not None:
            set_line_variant(n, lines, prec, -1)
