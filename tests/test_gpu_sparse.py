"""W-stacking bins and tiles with few points (k_grid_sparse, k_degrid_direct)
against the FP64 restatement: the w-planes where the gridder's 8 x 8 x 16-cell
blocks meet the edges of the grid, of the sort tiles, of the planes and of the
kernel widths, and the visibilities of tiles with one point to several units.

Tolerances: complex128 sums of FP64 products, kernel values exact to about
beta (at most 37) roundings, stay within 1e-12 (1e-11 for visibilities, which
carry the rounding of phases up to 1e4 radians); complex64 kernel values and
products carry FP32 offsets and rounding, 3e-6 as the dense path's tests."""
import numpy as np
import pytest

from oracle import oracle as O

from conftest import rel_l2, wst_case

pytestmark = pytest.mark.gpu

def spread_case(nrow, nx, ny, fov, wscale):
    """wst_case with u and v over the whole grid (footprints wrap at its
    edges) and |w| up to wscale / 2 wavelengths."""
    k = wst_case(nrow, nx, ny, fov)
    uvw = k["uvw"].copy()
    uvw[:, 0] /= k["xpix"]
    uvw[:, 1] /= k["ypix"]
    uvw[:, 2] *= wscale
    k["uvw"] = uvw
    return k


CASES = [
    # nrow, nx, ny, fov, eps, tile: grid sides in cells are about 2 nx, 2 ny
    (1, 16, 16, 5.0, 1e-5, 8),        # one point
    (40, 16, 16, 10.0, 0.2, 8),       # kernel width 2, a grid of 4 x 4 blocks
    (300, 25, 45, 10.0, 1e-4, 8),     # 50 x 90 cells: tiles of 2, partial blocks
    (300, 30, 36, 20.0, 1e-6, 16),    # 60 x 72: tiles of 4 and 8
    (500, 64, 64, 20.0, 1e-6, 32),    # blocks inside tiles of 32
    (2000, 125, 64, 10.0, 1e-5, 16),  # 250 x 128
    (3000, 512, 300, 3.0, 1e-5, 8),   # more than 2048 blocks: whole blocks per wave
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("single", [True, False])
def test_sparse_gridding_vs_oracle(gpu, case, single):
    torch = gpu
    from cugridder_amd import Context
    nrow, nx, ny, fov, eps, tile = case
    k = spread_case(nrow, nx, ny, fov, 1000.0)
    ctx = Context(stop_after=1, dense_min=0, tile_grid=tile)
    cdt, rdt = (torch.complex64, torch.float32) if single else (torch.complex128, torch.float64)
    ctx.ms2dirty(torch.tensor(k["uvw"], device="cuda"), torch.tensor(k["ms"], dtype=cdt, device="cuda"),
                 torch.tensor(k["wgt"], dtype=rdt, device="cuda"), nx, ny, fov, k["f0"], eps)
    got = ctx.grid_view(cdt).cpu().numpy()
    ms = k["ms"].astype("c8" if single else "c16").astype("c16")
    wgt = k["wgt"].astype("f4" if single else "f8").astype("f8")
    ref = O.ms2dirty_grid(k["uvw"], k["f0"], ms, wgt, nx, ny, fov, eps, single=single)
    assert rel_l2(got, ref) <= (3e-6 if single else 1e-12)


@pytest.mark.parametrize("eps", [1e-12, 1e-14, 1.2e-16])
def test_sparse_gridding_wide_kernels(gpu, eps):
    """Kernel widths 13, 15 and 16 (complex128 only), several windows of
    planes, a uv plane with crowded and empty blocks."""
    torch = gpu
    from cugridder_amd import Context
    k = spread_case(800, 60, 50, 25.0, 500.0)
    uvw = k["uvw"].copy()
    uvw[:500, :2] *= 0.05
    ctx = Context(stop_after=1)
    ctx.ms2dirty(torch.tensor(uvw, device="cuda"), torch.tensor(k["ms"], device="cuda"),
                 torch.tensor(k["wgt"], device="cuda"), 60, 50, 25.0, k["f0"], eps)
    got = ctx.grid_view(torch.complex128).cpu().numpy()
    ref = O.ms2dirty_grid(uvw, k["f0"], k["ms"], k["wgt"], 60, 50, 25.0, eps)
    assert rel_l2(got, ref) <= 1e-12


@pytest.mark.parametrize("case", CASES + [(4000, 40, 40, 10.0, 1e-5, 16),    # several units per tile
                                          (9000, 40, 40, 10.0, 1e-5, 16)])  # tiles above 256 points
@pytest.mark.parametrize("single", [True, False])
def test_direct_degridding_vs_oracle(gpu, case, single):
    torch = gpu
    from cugridder_amd import Context
    nrow, nx, ny, fov, eps, tile = case
    k = spread_case(nrow, nx, ny, fov, 1000.0)
    cdt, rdt = (torch.complex64, torch.float32) if single else (torch.complex128, torch.float64)
    dirty = k["dirty"].astype("f4" if single else "f8")
    wgt = k["wgt"].astype("f4" if single else "f8")
    ref = O.dirty2ms(k["uvw"], k["f0"], dirty.astype("c16"), wgt.astype("f8"), fov, eps, single=single)
    for slab in (0, 1):
        ctx = Context(tile_degrid=tile)
        if slab:
            plane = 4 * nx * ny * (8 if single else 16) * 1.2
            ctx.set_option("grid_limit_mb", max(1, int(plane * 3) >> 20))
        got = ctx.dirty2ms(torch.tensor(k["uvw"], device="cuda"), torch.tensor(dirty, dtype=cdt, device="cuda"),
                           torch.tensor(wgt, dtype=rdt, device="cuda"), fov, k["f0"], eps).cpu().numpy()
        assert rel_l2(got, ref) <= (3e-6 if single else 1e-11)


@pytest.mark.parametrize("eps", [1e-12, 1e-14, 1.2e-16])
def test_direct_degridding_wide_kernels(gpu, eps):
    torch = gpu
    from cugridder_amd import Context
    k = spread_case(800, 60, 50, 25.0, 500.0)
    got = Context().dirty2ms(torch.tensor(k["uvw"], device="cuda"),
                             torch.tensor(k["dirty"], dtype=torch.complex128, device="cuda"),
                             torch.tensor(k["wgt"], device="cuda"), 25.0, k["f0"], eps).cpu().numpy()
    ref = O.dirty2ms(k["uvw"], k["f0"], k["dirty"].astype("c16"), k["wgt"], 25.0, eps)
    assert rel_l2(got, ref) <= 1e-11
