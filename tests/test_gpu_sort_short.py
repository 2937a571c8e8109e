"""Short radix sorts (no scan launches): bit-exact against numpy's stable
sort where the tile size changes, with ragged last tiles, one to four passes,
crowded digits and a single key."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2, 255, 1024, 1025, 40000, 1 << 17, (1 << 17) + 1, 1 << 18, (1 << 18) + 1, (1 << 19) - 3,
                               (1 << 19) + 1])
@pytest.mark.parametrize("bits,crowd", [(8, 0), (13, 0), (22, 0.9), (32, 0.3), (24, 1.0)])
def test_short_sort(gpu, m, bits, crowd):
    torch = gpu
    from cugridder_amd import Context
    rng = np.random.default_rng(m * 37 + bits)
    keys = rng.integers(0, 1 << bits, size=m, dtype=np.uint64).astype(np.uint32)
    keys[rng.random(m) < crowd] = keys[0]
    tk = torch.tensor(keys.view(np.int32), device="cuda")
    tv = torch.arange(m, dtype=torch.int32, device="cuda")
    ctx = Context()
    ctx.sort_pairs(tk, tv, bits)
    ref = np.argsort(keys, kind="stable")
    assert np.array_equal(tv.cpu().numpy(), ref)
    assert np.array_equal(tk.cpu().numpy().view(np.uint32), keys[ref])
