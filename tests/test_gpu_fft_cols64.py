"""complex128 column steps of powers of two by both kernels: transforms below and
above a gibibyte and with sub-transforms of 16 to 128 points against numpy.fft,
and whole calls with the rows no point reaches left out against the same calls
with every row."""
import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


# (planes, columns' length, rows' length); 64 columns more than a gibibyte holds
@pytest.mark.parametrize("shape", [(1, 256, 2), (3, 256, 90), (2, 512, 30), (1, 1024, 512), (2, 2048, 72),
                                   (1, 4096, 36), (1, 8192, 40), (1, 16384, 6), (257, 256, 1024),
                                   (17, 2048, 2048), (17, 4096, 1024)])
def test_columns(gpu, shape):
    torch = gpu
    from cugridder_amd import Context
    b, n2, n1 = shape
    g = torch.Generator(device="cuda")
    g.manual_seed(n1 + n2)
    x = torch.view_as_complex(torch.randn(b, n2, n1, 2, generator=g, device="cuda", dtype=torch.float64))
    # log2(n1 n2) levels of about three roundings of half an ulp each
    tol = 1.5 * np.sqrt(np.log2(n1 * n2)) * np.finfo(np.float64).eps
    ctx = Context()
    for d in (1, -1):
        y = x.clone()
        ctx.fft2d(y, d)
        for p in {0, b // 2, b - 1}:
            z = x[p].cpu().numpy()
            ref = np.fft.ifft2(z) * (n1 * n2) if d == 1 else np.fft.fft2(z)
            assert rel_l2(y[p].cpu().numpy(), ref) < tol


@pytest.mark.parametrize("n,slab", [(128, 0), (256, 0), (512, 0), (1024, 0), (2048, 0), (512, 40)])
def test_masked_rows(gpu, n, slab):
    """Points near the centre only, after a call that left NaN in every plane."""
    torch = gpu
    from cugridder_amd import Context
    rng = np.random.default_rng(n)
    fov, f0 = 2.0, 1e9
    reach = 0.04 * n / np.radians(fov) * 0.299792458
    uvw = (rng.random((500, 3)) - 0.5) * 2 * reach
    uvw[:, 2] *= 0.02
    vis = torch.tensor(rng.standard_normal(500) + 1j * rng.standard_normal(500), device="cuda")
    img = torch.tensor(rng.standard_normal((n, n)) + 0j, device="cuda")
    full, near = torch.tensor(uvw * [11, 11, 1], device="cuda"), torch.tensor(uvw, device="cuda")
    out = []
    for mask in (0, 1):
        ctx = Context(row_mask=mask, grid_limit_mb=slab)
        ctx.ms2dirty(full, vis * float("nan"), None, n, n, fov, f0, 1e-6)
        a = ctx.ms2dirty(near, vis, None, n, n, fov, f0, 1e-6).cpu().numpy()
        ctx.ms2dirty(full, vis * float("nan"), None, n, n, fov, f0, 1e-6)
        b = ctx.dirty2ms(near, img, None, fov, f0, 1e-6).cpu().numpy()
        out.append((a, b))
        ctx.close()
    for a, b in zip(*out):
        # the same arithmetic on the same values: the masked cells are zero
        assert np.all(np.isfinite(a)) and rel_l2(b, a) < 1e-14
