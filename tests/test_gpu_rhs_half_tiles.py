"""The point operator's tiles of half the lanes (k_rhs) at their edges: rows of
one tile, of a whole one and a point more or less, of two and three, and the
rows where tiles of the full width take over and give way again.  The check and
its tolerance are test_gpu_rhs's; a staged batch, whose tiles have the full
width, gives the same bits."""
import pytest

from tests.test_gpu_rhs import KINDS, test_point_operator_tiles as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", KINDS, ids=[" ".join(f"{k}{v}" for k, v in c.items()) or "plain" for c in KINDS])
@pytest.mark.parametrize("nx,ny", [(42, 8), (43, 9), (44, 8), (85, 9), (86, 8), (87, 9), (128, 8), (129, 9), (130, 8),
                                   (172, 9), (173, 8), (258, 9)])
def test_half_tiles(orc, nx, ny, kw):
    check(orc, nx, ny, kw)


def test_half_tiles_have_the_bits_of_full_ones():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from lns3d_amd.batch import Batch
    from lns3d_amd.config import Params
    from lns3d_amd.native import MODE_BATCHED
    params = [Params(nx=nx, ny=ny, kz=0.3) for nx, ny in ((43, 9), (44, 21), (87, 17), (95, 33), (129, 65))] + \
             [Params(nx=100, ny=20, kz=0.4, xper=1, periodic_exact=1)]
    b = Batch(params, precision=1, seed=4)
    for k in range(len(params)):
        b.run_eager(k, 2)
    torch.cuda.synchronize()
    want = [v.clone() for v in b.v]
    b.reset()
    g = b.capture(2, MODE_BATCHED, 1)
    g.launch()
    g.synchronize()
    for k, (v, w) in enumerate(zip(b.v, want)):
        assert torch.equal(v, w), k
    g.close()
    b.close()
