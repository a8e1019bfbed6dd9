"""The line factorisation (k_factor_chains) where its register path begins and
ends: lines too short for it, with one and a few interior pivots, plain and
twisted, pivots whose larger part is the imaginary one, and pivots near the
ends of the exponent range, which are divided by in full.

Against a dense solve in complex double.  Tolerance: an elimination's rounding
is at most about 25 n eps relative to the solution times the lines' condition,
which their diagonals (2.0 and up over couplings of 0.3) keep below 20."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def columns(i, n):
    lo = 0 if i < 2 else n - 5 if i > n - 3 else i - 2
    return [lo + (i - 2 + k - lo) % 5 for k in range(5)]


@pytest.mark.parametrize("turn,scale", [(1.0, 1.0), (1j, 1.0), (1.0, 1e-130), (1j, 1e130)])
@pytest.mark.parametrize("lines,n", [(2, 7), (2, 8), (2, 9), (2, 15), (2, 16), (2, 17), (2, 18), (2, 21), (3, 64),
                                     (514, 9), (513, 16), (514, 33)])
def test_factor(lines, n, turn, scale):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lns3d_amd.native import Penta
    print(f"factor lines={lines} n={n} turn={turn} scale={scale}", flush=True)
    rng = np.random.default_rng(100 * n + lines)
    cplx = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    mat = 0.1 * cplx(lines, n, 5, 5, 5)              # [line][row][column][row of block][slot]
    for c in range(5):
        mat[:, :, c, c, 2] += 2.0 + 0.5 * c
    mat *= turn * scale
    rhs = scale * cplx(lines, n, 5)
    h = Penta(0, 2, lines, n)
    x = torch.from_numpy(rhs).cuda()
    h.factor(torch.from_numpy(mat).cuda())
    h.solve(x)
    x = x.cpu().numpy()
    for line in {0, 1, lines - 1}:
        a = np.zeros((5 * n, 5 * n), complex)
        for i in range(n):
            for k, c in enumerate(columns(i, n)):
                a[5 * i:5 * i + 5, 5 * c:5 * c + 5] = mat[line, i, :, :, k].T / scale
        ref = np.linalg.solve(a, rhs[line].reshape(-1) / scale)
        assert abs(x[line].reshape(-1) - ref).max() < 25 * n * 2.2e-16 * 20 * abs(ref).max()
    h.close()
