"""W-stacking degridding with few and many points per tile in one call: tiles read
straight from the planes (k_degrid_direct), tiles staged whole (k_degrid) and dense
bins, against the FP64 restatement.  Outputs start as NaN, so that a row that no
kernel writes shows.

Tolerances: the same sums in another order, 1e-11 relative in complex128 and FP32
rounding (3e-6) in complex64, as in test_gpu_sparse.py."""
import numpy as np
import pytest

from oracle import oracle as O

from conftest import rel_l2, wst_case

pytestmark = pytest.mark.gpu


def counted_case(nx, fov, kw, tile, counts, rest, wscale):
    """counts[i] points whose footprints begin in tile (3, 2 + 2 i) of a grid of
    2 nx cells a side, `rest` points over the tile rows from 5 on."""
    nrow = sum(counts) + rest
    k = wst_case(nrow, nx, nx, fov)
    rng = np.random.default_rng(nx + kw)
    cell = 1 / (2 * nx * k["xpix"]) * 299792458.0 / k["f0"]
    pos = rng.uniform(-0.9 * nx, 0.9 * nx, (nrow, 2))
    pos[:, 0] = rng.uniform(5 * tile + kw - nx, 0.9 * nx, nrow)
    at = 0
    for i, n in enumerate(counts):
        lo = np.array([3, 2 + 2 * i]) * tile + kw / 2 - nx
        pos[at:at + n] = lo + rng.uniform(0.2, 0.8, (n, 2)) * tile
        at += n
    uvw = np.empty((nrow, 3))
    uvw[:, :2] = pos * cell
    uvw[:, 2] = rng.uniform(-0.5, 0.5, nrow) * wscale * 299792458.0 / k["f0"]
    order = rng.permutation(nrow)
    k["uvw"] = uvw[order]
    return k


CASES = [
    # nx, eps, tile, kw, counts per crowded tile, other points
    (256, 1e-5, 16, 6, (255, 256, 257, 1500, 1), 4000),   # threshold 256, tiles of many units
    (128, 1e-3, 8, 4, (255, 256, 257, 4000, 40), 6000),   # the same on tiles of 8
    (150, 1e-8, 4, 9, (94, 95, 96, 97, 700), 5000),       # 300 cells: tiles of 4, threshold 96
    (125, 1e-6, 2, 7, (71, 72, 73, 74, 500), 5000),       # 250 cells: tiles of 2, threshold 72
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("single", [True, False])
def test_mixed_tiles_vs_oracle(gpu, case, single):
    torch = gpu
    from cugridder_amd import Context
    nx, eps, tile, kw, counts, rest = case
    if single and eps < 1e-6:
        pytest.skip("complex64 does not reach it")
    fov, wscale = 15.0, 400.0
    k = counted_case(nx, fov, kw, tile, counts, rest, wscale)
    cdt, rdt = (torch.complex64, torch.float32) if single else (torch.complex128, torch.float64)
    np_r = "f4" if single else "f8"
    dirty, wgt = k["dirty"].astype(np_r), k["wgt"].astype(np_r)
    ref = O.dirty2ms(k["uvw"], k["f0"], dirty.astype("c16"), wgt.astype("f8"), fov, eps, single=single)
    args = (torch.tensor(k["uvw"], device="cuda"), torch.tensor(dirty, dtype=cdt, device="cuda"),
            torch.tensor(wgt, dtype=rdt, device="cuda"), fov, k["f0"], eps)
    opts = [dict(), dict(grid_limit_mb=max(1, int(4 * nx * nx * (8 if single else 16) * 9) >> 20))]
    if single:
        opts.append(dict(degrid_dense_min=0))
    for o in opts:
        ctx = Context(tile_degrid=tile, **o)
        out = torch.full((len(k["uvw"]),), complex("nan"), dtype=cdt, device="cuda")
        got = ctx.dirty2ms(*args, out=out).cpu().numpy()
        assert ctx.last_plan()["kw"] == kw
        if "grid_limit_mb" in o:
            assert ctx.last_slab()[1] >= 2
        assert rel_l2(got, ref) <= (3e-6 if single else 1e-11), o
