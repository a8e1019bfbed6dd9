"""A non-finite field in the refined steps: the residual's norms keep a NaN
(or an infinity) that any one of their values holds, so the adaptive step
reports it and leaves v as it was, and the fixed step's residual is not a
number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _step(nx, ny, **kw):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lns3d_amd.config import Params, make_disturbance, make_grid, make_mean
    from lns3d_amd.native import Step
    p = Params(nx=nx, ny=ny, kz=0.3, **kw)
    x, y, met = make_grid(p)
    st = Step(p, precision=1)
    st.setup(met, make_mean(p, y))
    st.factor()
    v = torch.from_numpy(np.ascontiguousarray(make_disturbance(p, x, seed=6).reshape(-1, order="F"))).to("cuda")
    st.itrbc3d(v)
    return torch, st, v


# where: one value of the field (the first and last wave of the operator's
# workgroups, a place between), or all of it
@pytest.mark.parametrize("bad", [complex(np.nan, 0), complex(0, np.nan), complex(np.inf, 0), complex(0, -np.inf)])
@pytest.mark.parametrize("nx,ny,kw,where", [(33, 17, {}, (16, 8)), (65, 33, {}, (2, 1)), (65, 33, {}, (62, 31)),
                                            (33, 17, {}, None), (33, 17, dict(xper=1, periodic_exact=1), (5, 9))])
def test_refined_step_reports_nonfinite(nx, ny, kw, where, bad):
    from lns3d_amd.native import LNS3DError, ENONFINITE
    print(f"non-finite {nx}x{ny} {kw} {where} {bad}", flush=True)
    torch, st, v = _step(nx, ny, **kw)
    if where is None:
        v.fill_(bad)
    else:
        v.reshape(ny, nx, 5)[where[1], where[0], 2] = bad
    bits = torch.view_as_real(v).view(torch.int64).clone()
    with pytest.raises(LNS3DError) as e:
        st.step_refined(v, torch.zeros_like(v), tol=1e-10, max_iters=8)
    assert e.value.code == ENONFINITE
    assert torch.equal(torch.view_as_real(v).view(torch.int64), bits)
    assert not np.isfinite(st.last_residual())
    # the form without a host synchronisation, with the check and without
    for check in (True, False):
        w = v.clone()
        st.step_refined_fixed(w, torch.zeros_like(w), 1, check)
        assert not np.isfinite(st.last_residual())
    st.close()


def test_refined_step_zero_field_is_finite():
    """no residual at all is 0, not a number over zero"""
    torch, st, v = _step(33, 17)
    v.zero_()
    its, res = st.step_refined(v, torch.zeros_like(v), tol=1e-10, max_iters=8)
    assert (its, res, st.last_residual()) == (1, 0.0, 0.0)
    assert not bool(v.abs().max())
    st.close()
