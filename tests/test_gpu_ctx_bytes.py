"""lns3d_ctx_bytes against the device memory that a factored context takes, by
which the serving loop admits requests.

Tolerance: a context makes fewer than 32 allocations, each rounded up to a
page of 2 MiB at most."""
import gc

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kw", [{}, dict(xper=1), dict(yper=1), dict(xper=1, yper=1), dict(Re=0.0),
                                dict(nx=2049, ny=65)],
                         ids=lambda kw: " ".join(f"{k}{v}" for k, v in kw.items()) or "plain")
def test_ctx_bytes(kw, precision):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lns3d_amd.config import Params, make_grid, make_mean
    from lns3d_amd.native import Step, ctx_bytes
    print(f"ctx bytes {kw} precision={precision}", flush=True)
    p = Params(**dict(dict(nx=513, ny=257, kz=0.3, periodic_exact=1), **kw))
    x, y, met = make_grid(p)
    vm = make_mean(p, y)
    for measured in (False, True):     # the first one brings in the kernels' own memory
        gc.collect()                   # contexts that other tests left behind give theirs back here, not below
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        st = Step(p, precision=precision)
        st.setup(met, vm)
        st.factor()
        torch.cuda.synchronize()
        taken = before - torch.cuda.mem_get_info()[0]
        st.close()
    said = ctx_bytes(p, precision)
    print(f"  taken {taken / 2**20:.1f} MiB, said {said / 2**20:.1f}", flush=True)
    assert -2**20 <= taken - said <= 32 * 2**21
