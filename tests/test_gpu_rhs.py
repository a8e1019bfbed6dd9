"""The point operator's tiles (k_rhs) at their edges: rows of one tile, of a
whole tile and a point more or less, of two and three tiles; rows too short
for an interior point; periodic rows whose last column is no copy of the
first; symmetric ends.  Against the oracle's lrhs3D on white noise.

Tolerance: U_xieta is a sum of 36 products taken in another order than the
oracle's, a few units of rounding of terms no larger than the operator's
values on white noise: 1e-12 of the largest value leaves a factor of 1000,
which the coefficients' own rounding differences share."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(7, 7), (8, 13), (93, 8), (94, 7), (95, 9), (187, 8), (188, 9), (189, 7), (283, 11)]
KINDS = [dict(), dict(optx=0, opty=1, wallt=1), dict(xper=1, periodic_exact=1, wallt=2), dict(yper=1, periodic_exact=1),
         dict(xper=1, yper=1, periodic_exact=1), dict(left=7, right=7)]


@pytest.mark.parametrize("kw", KINDS, ids=[" ".join(f"{k}{v}" for k, v in c.items()) or "plain" for c in KINDS])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_point_operator_tiles(orc, nx, ny, kw):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lns3d_amd.config import Params, make_grid, make_mean
    from lns3d_amd.native import Step
    if kw.get("left") == 7 and nx < ny + 2:
        pytest.skip("symmetric ends need nx >= ny")
    if (kw.get("xper") and nx < 8) or (kw.get("yper") and ny < 8):
        pytest.skip("a periodic line has at least 7 unknowns, 8 points")
    print(f"rhs {nx}x{ny} {kw}", flush=True)
    p = Params(nx=nx, ny=ny, kz=0.4, **kw)
    x, y, met = make_grid(p)
    vm = make_mean(p, y)
    st = Step(p)
    st.setup(met, vm)
    co = orc.genmtrx(p, vm, met)
    rng = np.random.default_rng(nx * 31 + ny)
    v = np.asfortranarray(rng.standard_normal((5, nx, ny)) + 1j * rng.standard_normal((5, nx, ny)))
    want, _ = orc.lrhs3d(p, co, v)
    vd = torch.from_numpy(np.ascontiguousarray(v.reshape(-1, order="F"))).to("cuda")
    rd = torch.zeros_like(vd)
    st.lrhs3d(vd, rd)
    got = rd.cpu().numpy().reshape(v.shape, order="F")
    assert np.abs(got - want).max() < 1e-12 * np.abs(want).max()
    st.close()
