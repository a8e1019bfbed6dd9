"""The streaming solve of periodic lines at its edges: one and two lines a
workgroup, chains (rows less the last two) of fewer rows than a chunk, of
whole chunks and a row more or less, right-hand sides that stay in LDS or go
through its ring.  Against the oracle's cpenta_p.

Tolerances: diagonally dominant lines, a few units of rounding a row (1e-12
in complex double); complex-float records carry 6e-8 each, 1e-5 over the
lines' effective coupling length."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (lines, stored rows); unknowns are one fewer, the chain three fewer
EDGES = [(1 + n % 3, n) for n in (8, 9, 10, 14, 15, 16, 20, 21, 22, 26, 27, 28, 32, 33, 38, 39, 40, 51)]
SHAPES = [(3, 500), (3, 640), (2, 900), (513, 40), (514, 27), (515, 64), (513, 130)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("lines,n", EDGES + SHAPES)
def test_periodic_forms(orc, lines, n, prec):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lns3d_amd.native import Penta
    from tests.penta_cases import random_lines, relerr
    layout, exact = 1 + n % 2, (n // 2) % 2
    print(f"periodic form lines={lines} n={n} prec={prec} exact={exact}", flush=True)
    mat, rhs = random_lines(lines, n, layout, seed=5 * lines + n)
    m_ref, x_ref = mat.copy(order="F"), rhs.copy(order="F")
    shape = (2, 5, 5) + mat.shape[3:]
    per, per2 = np.zeros(shape, complex, order="F"), np.zeros(shape, complex, order="F")
    orc.cpenta_p(layout, m_ref, x_ref, per, per2, 2, exact)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.reshape(-1, order="F"))).to("cuda")
    h = Penta(1, layout, lines, n, prec, exact)
    dm, dr = dev(mat), dev(rhs)
    h.factor(dm)
    for _ in range(2):          # a second solve finds the LDS as the first left it
        dr.copy_(dev(rhs))
        h.solve(dr)
    assert relerr(dr.cpu().numpy().reshape(rhs.shape, order="F"), x_ref) < (1e-12 if prec == 0 else 1e-5)
    h.close()
