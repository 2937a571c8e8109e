"""W-stacking gridding with points crowded into a few tiles and no dense path:
the regions that go to k_grid instead of k_grid_sparse, the blocks beside them
and the tiles both write, against the FP64 restatement; and the time of such a
call, which a single wave per block made up to ten times longer.

Tolerances as in test_gpu_sparse.py."""
import time

import numpy as np
import pytest

from oracle import oracle as O

from conftest import rel_l2, wst_case

pytestmark = pytest.mark.gpu


def crowded_case(nrow, nx, ny, fov, wscale, at):
    """nrow rows within about two cells of (at) cells off the centre, a tenth of
    them over the whole grid, |w| up to wscale / 2 wavelengths."""
    k = wst_case(nrow, nx, ny, fov)
    rng = np.random.default_rng(nx + ny)
    uvw = k["uvw"].copy()
    uvw[:, 0] /= k["xpix"]
    uvw[:, 1] /= k["ypix"]
    uvw[:, 2] *= wscale
    near = np.arange(nrow) % 10 != 0
    # one grid cell is half a pixel's frequency: 1 / (2 nx xpix) wavelengths
    cell = np.array([1 / (2 * nx * k["xpix"]), 1 / (2 * ny * k["ypix"])]) * 299792458.0 / k["f0"]
    off = rng.uniform(-2, 2, (nrow, 2)) + np.asarray(at)
    uvw[near, :2] = (off * cell)[near]
    k["uvw"] = uvw
    return k


CASES = [
    # nrow, nx, ny, fov, |w| scale, eps, tile, cluster; grid sides about 2 nx, 2 ny
    (3000, 64, 64, 20.0, 300.0, 0.2, 8, (0, 0)),          # kernel width 2
    (3000, 64, 96, 20.0, 300.0, 1e-3, 8, (3, -5)),        # 128 x 192, tiles of 8
    (4000, 25, 45, 10.0, 300.0, 1e-4, 8, (-1, 2)),        # 50 x 90: tiles of 2, partial blocks
    (4000, 30, 36, 20.0, 300.0, 1e-5, 8, (10, 4)),        # 60 x 72: tiles of 4 and 8
    (6000, 64, 64, 20.0, 300.0, 1e-6, 8, (1, 1)),         # width 7
    (9000, 25, 45, 10.0, 300.0, 1e-7, 8, (0, 0)),         # width 8 on tiles of 2
    (3000, 64, 64, 20.0, 300.0, 1e-3, 32, (20, 9)),       # regions of 32
    (3000, 64, 64, 20.0, 300.0, 1e-3, 16, (-60, 58)),     # wraps past the edges
    (3000, 64, 96, 20.0, 300.0, 1e-3, 4, (0, 7)),         # tiles inside a block
    (20000, 40, 40, 40.0, 3000.0, 1e-2, 8, (2, 2)),       # many planes: windows and chunks
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("single", [True, False])
def test_crowded_gridding_vs_oracle(gpu, case, single):
    torch = gpu
    from cugridder_amd import Context
    nrow, nx, ny, fov, ws, eps, tile, at = case
    k = crowded_case(nrow, nx, ny, fov, ws, at)
    cdt, rdt = (torch.complex64, torch.float32) if single else (torch.complex128, torch.float64)
    args = (torch.tensor(k["uvw"], device="cuda"), torch.tensor(k["ms"], dtype=cdt, device="cuda"),
            torch.tensor(k["wgt"], dtype=rdt, device="cuda"), nx, ny, fov, k["f0"], eps)
    ms = k["ms"].astype("c8" if single else "c16").astype("c16")
    wgt = k["wgt"].astype("f4" if single else "f8").astype("f8")
    ref = O.ms2dirty_grid(k["uvw"], k["f0"], ms, wgt, nx, ny, fov, eps, single=single)
    tol = 3e-6 if single else 1e-12
    ctx = Context(stop_after=1, dense_min=0, tile_grid=tile)
    # cells no kernel writes would stay NaN
    ctx.ms2dirty(args[0] * 0.999, args[1] * float("nan"), *args[2:])
    ctx.ms2dirty(*args)
    assert rel_l2(ctx.grid_view(cdt).cpu().numpy(), ref) <= tol
    # the whole call with the rows and columns no point reaches left out, and in
    # slabs of planes
    img = []
    for opts in (dict(row_mask=0), dict(row_mask=1), dict(grid_limit_mb=1)):
        ctx = Context(dense_min=0, tile_grid=tile, **opts)
        ctx.ms2dirty(args[0] * 0.999, args[1] * float("nan"), *args[2:])
        img.append(ctx.ms2dirty(*args).cpu().numpy())
    for i in img[1:]:
        assert rel_l2(i, img[0]) <= tol


def test_crowded_call_is_not_serial(gpu):
    """10^5 complex128 rows within two cells take about five times as long as
    spread over the grid (1.1 against 0.23 ms); one wave's chain took 40 times."""
    torch = gpu
    from cugridder_amd import Context
    n, nx, fov, f0 = 100000, 512, 2.0, 1e9
    rng = np.random.default_rng(3)
    cell = 299792458.0 / f0 / (2 * np.radians(fov))
    ctx = Context()
    vis = torch.ones(n, dtype=torch.complex128, device="cuda")
    ms = []
    for spread in (1.0, 150.0):
        uvw = np.clip(rng.standard_normal((n, 3)) * spread, -450, 450) * cell
        uvw[:, 2] = rng.uniform(-100, 100, n) * 299792458.0 / f0
        t = torch.tensor(uvw, device="cuda")
        best = []
        for _ in range(8):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            ctx.ms2dirty(t, vis, None, nx, nx, fov, f0, 0.1)
            torch.cuda.synchronize()
            best.append(time.perf_counter() - t0)
        ms.append(min(best) * 1e3)
    assert ms[0] < 12 * ms[1], ms


def test_crowded_batch_replays(gpu):
    """Channels with crowded regions captured as one graph (complex64, several windows
    of planes, so no dense path): every replay gives the single call's image, with
    eager calls between the replays."""
    torch = gpu
    from cugridder_amd import Context
    ctx = Context()
    items, ref = [], []
    for nx, ny, n in ((64, 64, 20000), (30, 36, 6000)):
        k = crowded_case(n, nx, ny, 40.0, 2000.0, (1, -2))
        it = dict(uvw=torch.tensor(k["uvw"], device="cuda"),
                  vis=torch.tensor(k["ms"], dtype=torch.complex64, device="cuda"),
                  wgt=torch.tensor(k["wgt"], dtype=torch.float32, device="cuda"), fov=40.0, freq=k["f0"],
                  dirty=torch.zeros(nx, ny, dtype=torch.complex64, device="cuda"))
        items.append(it)
        ref.append(ctx.ms2dirty(it["uvw"], it["vis"], it["wgt"], nx, ny, 40.0, k["f0"], 1e-2).cpu().numpy())
        assert ctx.last_plan()["nf3"] > 32
    batch = ctx.batch("ms2dirty", items, 1e-2, graph=True)
    for _ in range(4):
        for it in items:
            it["dirty"].fill_(5.0)
        batch.run()
        torch.cuda.synchronize()
        for it, r in zip(items, ref):
            assert rel_l2(it["dirty"].cpu().numpy(), r) < 2e-6
        ctx.ms2dirty(items[0]["uvw"], items[0]["vis"], None, 64, 64, 40.0, items[0]["freq"], 1e-2)
