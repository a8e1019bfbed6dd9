"""The end of a step (v += dv and the boundary conditions in one kernel)
against its parts: the new field is bit for bit lns3d_itrbc3d, the boundary
kernels by themselves, of the old field plus the increment the step returns
(both are one rounded addition per part, so there is no tolerance).

Sizes at the edges: the smallest grid, fewer and more values in a row than a
workgroup, wall strips of one and five rows, partial wall extents."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    dict(nx=7, ny=7), dict(nx=7, ny=7, wall=1, wallt=1), dict(nx=64, ny=8, wall=2, wallt=2),
    dict(nx=53, ny=9, wall=1, wallt=0, wall_is=5, wall_ie=40), dict(nx=51, ny=11, wall=0, wallt=1),
    dict(nx=40, ny=20, wall=3, wallt=0, wall_is=3, wall_ie=38), dict(nx=40, ny=20, wall=3, wallt=1),
    dict(nx=33, ny=17, xper=1, periodic_exact=1, wall=1, wallt=1), dict(nx=33, ny=17, yper=1, periodic_exact=1),
    dict(nx=33, ny=17, xper=1, yper=1, periodic_exact=1), dict(nx=65, ny=33, top=1, left=1),
    dict(nx=30, ny=40, left=5, right=5, wall=2), dict(nx=48, ny=24, left=7, right=7, wall=1, wallt=1),
    dict(nx=31, ny=13, right=9, wall=1, wallt=1), dict(nx=31, ny=13, right=8, left=7),
    dict(nx=45, ny=15, Re=0.0, wall_is=4, wall_ie=41), dict(nx=45, ny=15, Re=0.0, right=9),
    dict(nx=45, ny=15, Re=0.0, xper=1, periodic_exact=1),
]


@pytest.mark.parametrize("form", ["step", "refined1", "refined2"])
@pytest.mark.parametrize("kw", CASES, ids=[" ".join(f"{k}{v}" for k, v in c.items()) for c in CASES])
def test_update_is_its_parts(kw, form):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lns3d_amd.config import Params, make_disturbance, make_grid, make_mean
    from lns3d_amd.native import Step
    print(f"update {kw} {form}", flush=True)
    p = Params(kz=0.3, **kw)
    x, y, met = make_grid(p)
    st = Step(p, precision=int(form != "step"))
    st.setup(met, make_mean(p, y))
    rng = np.random.default_rng(5)
    xg = np.asfortranarray(np.broadcast_to(np.asarray(x).reshape(p.nx, -1)[:, :1], (p.nx, p.ny)))
    if p.wall == 3:
        st.set_wall(rng.standard_normal((p.nx, 5)) + 1j * rng.standard_normal((p.nx, 5)))
    if p.top == 1:
        st.set_top_forcing(xg)
    if p.left in (1, 5) or p.right == 5:
        st.set_inflow(xg, 0.0)
    st.factor()
    v = torch.from_numpy(np.ascontiguousarray(make_disturbance(p, x, seed=3).reshape(-1, order="F"))).to("cuda")
    v += 1e-3 * torch.from_numpy(rng.standard_normal(v.numel()) + 1j * rng.standard_normal(v.numel())).to("cuda")
    st.itrbc3d(v)
    dv = torch.zeros_like(v)
    for _ in range(2):
        old = v.clone()
        if form == "step":
            st.step(v, dv)
        else:
            st.step_refined_fixed(v, dv, int(form[-1]))
        want = old + dv
        st.itrbc3d(want)
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(v).view(torch.int64), torch.view_as_real(want).view(torch.int64))
        assert not torch.equal(v, old)
    st.close()
