"""Mixed-radix FFT passes (lengths 2^a 3^b 5^c): the plane transform against
FP64 torch.fft on the host, and whole calls on grids of such sides, whose masked
rows, masked columns and dead frequencies are neither read nor written, against
the same calls without the masks."""
import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

# (planes, columns' length, rows' length): every radix alone and in products,
# whole columns (<= 128) and split ones, several rows per workgroup, blocks of
# fewer than 64 columns, the longest rows
SHAPES = [(1, 2, 2), (3, 6, 10), (2, 9, 12), (1, 15, 20), (2, 25, 16), (1, 5, 27), (1, 54, 50), (2, 60, 96),
          (3, 120, 75), (1, 125, 324), (1, 128, 250), (2, 150, 192), (1, 192, 256), (1, 486, 100), (1, 500, 3000),
          (2, 2500, 90), (1, 3000, 36), (1, 4800, 6), (1, 50, 4374), (1, 30, 6250), (1, 20, 7776), (1, 40, 7290)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
def test_mixed_fft2d(gpu, shape, dtype):
    torch = gpu
    from cugridder_amd import Context
    b, n2, n1 = shape
    rng = np.random.default_rng(n1 + 7 * n2)
    x = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(dtype)
    ctx = Context()
    # each of log2(n1 n2) levels rounds its sums and one twiddle product: about
    # three roundings of half an ulp, adding in quadrature over the levels
    tol = 1.5 * np.sqrt(np.log2(n1 * n2)) * np.finfo(dtype).eps
    for d in (1, -1):
        y = torch.tensor(x, device="cuda")
        ctx.fft2d(y, d)
        z = x.astype(np.complex128)
        ref = np.fft.ifft2(z) * (n1 * n2) if d == 1 else np.fft.fft2(z)
        assert rel_l2(y.cpu().numpy(), ref) < tol


@pytest.mark.parametrize("nx,ny", [(33, 60), (60, 250), (96, 1250), (1250, 96), (1500, 90), (625, 375)])
@pytest.mark.parametrize("double", [False, True])
def test_masks_on_mixed_sizes(gpu, nx, ny, double):
    """Rows and columns no point reaches change nothing, whatever the buffer
    held: a few points near the centre, after a call that filled the grid."""
    torch = gpu
    from cugridder_amd import Context
    rng = np.random.default_rng(nx * 3 + ny)
    c, r = (np.complex128, np.float64) if double else (np.complex64, np.float32)
    eps = 1e-9 if double else 1e-5
    fov, f0 = 2.0, 1e9
    reach = 0.04 * nx / np.radians(fov) * 0.299792458
    n = 700
    uvw = (rng.random((n, 3)) - 0.5) * 2 * reach
    uvw[:, 1] *= ny / nx
    vis = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(c)
    img = rng.standard_normal((nx, ny)).astype(c)
    wgt = (rng.random(n) + 0.5).astype(r)
    full = torch.tensor(uvw * 11, device="cuda")
    tu, tv = torch.tensor(uvw, device="cuda"), torch.tensor(vis, device="cuda")
    ti, tw = torch.tensor(img, device="cuda"), torch.tensor(wgt, device="cuda")
    out = {}
    for mask in (0, 1):
        ctx = Context(row_mask=mask)
        # leaves NaN in every plane
        ctx.ms2dirty(full, tv * float("nan"), tw, nx, ny, fov, f0, eps)
        a = ctx.ms2dirty(tu, tv, tw, nx, ny, fov, f0, eps).cpu().numpy()
        ctx.ms2dirty(full, tv * float("nan"), tw, nx, ny, fov, f0, eps)
        b = ctx.dirty2ms(tu, ti, tw, fov, f0, eps).cpu().numpy()
        out[mask] = (a, b)
        ctx.close()
    for a, b in zip(out[1], out[0]):
        assert np.all(np.isfinite(a))
        # the same arithmetic on the same values: the masked cells are zero
        assert rel_l2(a, b) < (1e-14 if double else 1e-6)
