"""Routes of the complex-float steps that only some shapes and decks take, bit
for bit.

* The first solve of a refined step reads the residual and leaves the increment
  elsewhere: without corrections that is the complex-float step, whose solve is
  in place.  Every form of the line solve that a context reaches: plain lines
  with resident right-hand sides and a ring, twisted lines, periodic lines with
  resident right-hand sides of both chunk lengths and a ring.
* right = 9 reads two columns inside it, so a kernel of its own follows the
  update: in a staged graph it has workgroups for those members only."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(torch, t):
    return torch.view_as_real(t).view(torch.int64)


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("nx,ny,xper", [(100, 520, 0), (90, 1030, 0), (150, 1601, 0), (384, 520, 0), (129, 65, 0),
                                        (700, 9, 1), (150, 521, 1), (300, 513, 1), (40, 20, 1), (200, 40, 1)])
def test_out_of_place_first_solve(nx, ny, xper):
    from lns3d_amd.config import Params, make_disturbance, make_grid, make_mean
    from lns3d_amd.native import Step
    torch = _torch()
    print(f"out of place {nx}x{ny} xper={xper}", flush=True)
    p = Params(nx=nx, ny=ny, kz=0.3, xper=xper, periodic_exact=1)
    x, y, met = make_grid(p)
    st = Step(p, precision=1)
    st.setup(met, make_mean(p, y))
    st.factor()
    va = torch.from_numpy(np.ascontiguousarray(make_disturbance(p, x, seed=7).reshape(-1, order="F"))).to("cuda")
    st.itrbc3d(va)
    vb = va.clone()
    da, db = torch.zeros_like(va), torch.full_like(va, complex(np.nan, np.nan))
    for _ in range(2):
        st.step_fp32(va, da)
        st.step_refined_fixed(vb, db, 0)
        torch.cuda.synchronize()
        assert bool(torch.isfinite(_bits(torch, da).view(torch.float64)).all())
        assert torch.equal(_bits(torch, da), _bits(torch, db))
        assert torch.equal(_bits(torch, va), _bits(torch, vb))
    st.close()


@pytest.mark.parametrize("corrections", [0, 1, 2])
def test_staged_routes_match_branches(corrections):
    from lns3d_amd.batch import Batch
    from lns3d_amd.config import Params
    from lns3d_amd.native import Graph, MODE_BATCHED, MODE_FP32, MODE_REFINED
    torch = _torch()
    print(f"staged routes corrections={corrections}", flush=True)
    params = [Params(nx=150, ny=521, kz=0.3, xper=1, periodic_exact=1), Params(nx=700, ny=9, kz=0.3, xper=1),
              Params(nx=31, ny=13, kz=0.4, right=9, yper=1, periodic_exact=1), Params(nx=65, ny=33, kz=0.2),
              Params(nx=100, ny=520, kz=0.5), Params(nx=45, ny=19, kz=0.6, right=9, yper=1, periodic_exact=1)]
    b = Batch(params, precision=1, seed=2)
    rng = np.random.default_rng(3)
    for st, v, v0 in zip(b.steps, b.v, b.v0):       # right = 9 divides by the field: none of it is zero
        v += 1e-2 * torch.from_numpy(rng.standard_normal(v.numel()) + 1j * rng.standard_normal(v.numel())).cuda()
        st.itrbc3d(v)
        v0.copy_(v)
    out = []
    for mode in (MODE_REFINED if corrections else MODE_FP32, MODE_BATCHED):
        b.reset()
        torch.cuda.synchronize()
        g = Graph(b.steps, b.v, b.dv, nsteps=2, mode=mode, corrections=corrections)
        g.launch()
        g.synchronize()
        out.append([v.clone() for v in b.v + b.dv])
        g.close()
    for k, (a, c) in enumerate(zip(*out)):
        assert bool(torch.isfinite(_bits(torch, c).view(torch.float64)).all()), k
        assert torch.equal(_bits(torch, a), _bits(torch, c)), k
    b.close()
