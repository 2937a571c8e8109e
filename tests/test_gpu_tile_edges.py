"""ms2dirty with gridding tiles down to one cell: the same image as with the
default tiles."""
import pytest

from tests.conftest import rel_l2, wst_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 12])
@pytest.mark.parametrize("single", [True, False])
def test_small_tiles(gpu, tile, single):
    torch = gpu
    from cugridder_amd import Context
    k = wst_case(700, 40, 36, 15.0)
    uvw = k["uvw"].copy()
    uvw[:, 0] /= k["xpix"]
    uvw[:, 1] /= k["ypix"]
    cdt, rdt = (torch.complex64, torch.float32) if single else (torch.complex128, torch.float64)
    args = (torch.tensor(uvw, device="cuda"), torch.tensor(k["ms"], dtype=cdt, device="cuda"),
            torch.tensor(k["wgt"], dtype=rdt, device="cuda"), 40, 36, 15.0, k["f0"], 1e-5)
    ref = Context().ms2dirty(*args).cpu().numpy()
    got = Context(tile_grid=tile).ms2dirty(*args).cpu().numpy()
    # the same products in another order of the sums
    assert rel_l2(got, ref) < (3e-6 if single else 1e-13)
