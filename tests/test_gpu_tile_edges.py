"""Gridding tiles at their limits.  ms2dirty with tiles down to one cell: the same
image as with the default tiles.  nufft2d1 with one tile along an axis, where
footprints wrap inside the tile, against the FP64 restatement."""
import numpy as np
import pytest

from oracle import oracle as O
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


@pytest.mark.parametrize("single", [True, False])
@pytest.mark.parametrize("eps", [1e-2, 1e-5, 1e-7, 1e-12])
@pytest.mark.parametrize("N1,N2", [(16, 150), (150, 16), (16, 16), (60, 75)])
def test_one_tile_along_an_axis(gpu, N1, N2, eps, single):
    if single and eps < 1e-6:
        pytest.skip("complex64 does not reach it")
    torch = gpu
    from cugridder_amd import Context
    rng = np.random.default_rng(N1 + 7 * N2)
    M = 5000
    xy = rng.uniform(-np.pi, np.pi, (2, M))
    xy[:, ::3] = np.pi - np.abs(rng.normal(0, 0.05, xy[:, ::3].shape))   # crowded at the seam
    c = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    if single:
        xy, c = xy.astype("f4"), c.astype("c8")
        xy = np.clip(xy, np.float32(-3.14159), np.float32(3.14159))
    ref = O.nufft2d1(xy[0], xy[1], c, N1, N2, eps, single=single)
    t = [torch.from_numpy(a.copy()).cuda() for a in (xy[0], xy[1], c)]
    # the same terms in another order of the sums (FP32 terms in complex64)
    for tile in (32, 8):
        got = Context(mfma2d=0, tile_grid2d=tile).nufft2d1(*t, N1, N2, eps).cpu().numpy()
        assert rel_l2(got, ref) <= max(eps if eps > 1e-10 else 0, 3e-6 if single else 1e-12)
