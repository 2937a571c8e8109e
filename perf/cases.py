"""Timed cases of the framework's public entry points on one GPU.

Each case is a dict of plain values.  ``prepare`` makes what a user's program
holds before the call, ``run`` is one pass through the public entry points,
``exact`` the same outputs as a direct FP64 sum and ``work`` the bytes and
operations one pass cannot do without.

Kinds of case:
* ``image``: ms2dirty (visibilities -> image) or dirty2ms (image ->
  visibilities), on device tensors through a Context, or, with ``host``, on
  numpy arrays through the NIFTY-style functions ms2dirty / dirty2ms;
* ``nufft``: the 2-D NUFFT, type 1 (points -> modes), 2 (modes -> points) or
  both in turn;
* ``batch``: independent channels of mixed sizes run as one graph.

Visibility coverages: ``tracks`` (Earth-rotation synthesis of an antenna
array, in time order as a measurement set stores it, or ``shuffled``),
``gauss`` (a compact array, Gaussian u and v) and ``uniform`` (u and v
filling the whole grid, as the accuracy benchmarks of this method draw them).
"""
import math
import random

import numpy as np
import torch

import cugridder_amd as cg

C_LIGHT = 299792458.0
_ctx = []


def _context():
    """The program's one Context: its workspace is kept from call to call."""
    if not _ctx:
        _ctx.append(cg.Context())
    return _ctx[0]


# ------------------------------------------------------------------ cases

def _image(name, direction, rows, nx, ny, fov, freq, eps, coverage, **more):
    c = dict(kind="image", direction=direction, rows=rows, nx=nx, ny=ny, fov=fov, freq=freq, eps=eps,
             coverage=coverage, extent=5000.0, channels=1, double=False, uvw32=False, weights=True,
             wstacking=True, shuffled=False, host=False)
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one snapshot of a small array onto a small image: a self-calibration
        # or preview call, where the number of launches counts
        _image("snapshot_ms2dirty", "ms2dirty", 2000, 128, 96, 2.0, 1e9, 1e-5, "tracks", extent=800.0),
        # the numpy-in, numpy-out call of the NIFTY-style binding, complex128:
        # predicted visibilities of a rectangular image
        _image("host_dirty2ms", "dirty2ms", 20000, 250, 128, 10.0, 1e9, 1e-7, "uniform", double=True,
               host=True),
        # the plain one-channel workload of the benchmark, both directions:
        # gridding and predicting inside a deconvolution loop
        _image("plain_ms2dirty", "ms2dirty", 131072, 1024, 1024, 2.0, 1e8, 1e-5, "gauss", extent=3000.0),
        _image("plain_dirty2ms", "dirty2ms", 131072, 1024, 1024, 2.0, 1e8, 1e-5, "gauss", extent=3000.0),
        # several channels of a time-ordered observation into one image whose
        # sides are neither equal nor powers of two
        _image("channels_ms2dirty", "ms2dirty", 12288, 1500, 1250, 3.0, 1.2e9, 1e-4, "tracks",
               channels=16, extent=3000.0),
        # one channel predicted for FP32 coordinates without weights on an odd
        # rectangular image
        _image("ragged_dirty2ms", "dirty2ms", 1000003, 2310, 3125, 4.0, 1.4e9, 1e-5, "tracks",
               extent=4000.0, uvw32=True, weights=False),
        # full W-stacking, the benchmark's default workload, both directions
        # (|w| up to 5000 wavelengths)
        _image("full_ms2dirty", "ms2dirty", 1 << 27, 8192, 8192, 3.0, 1.4e9, 1e-6, "tracks",
               weights=False, shuffled=True, extent=7660.0),
        _image("full_dirty2ms", "dirty2ms", 1 << 27, 8192, 8192, 3.0, 1.4e9, 1e-6, "tracks",
               weights=False, shuffled=True, extent=7660.0),
        # complex128 at eps 1e-12 on a wide field, 1e6 rows over the whole uv
        # plane: the high-accuracy workload of the method
        _image("double_ms2dirty", "ms2dirty", 1000000, 2048, 2048, 10.0, 1e9, 1e-12, "uniform",
               double=True),
        _image("double_dirty2ms", "dirty2ms", 1000000, 2048, 2048, 10.0, 1e9, 1e-12, "uniform",
               double=True),
        # the benchmark's clustered 2-D points: both types of the transform
        # run in turn by an iterative solver
        dict(kind="nufft", name="nufft2d_clustered", type="both", points=1 << 25, n1=4096, n2=4096, eps=1e-5,
             double=False, clustered=True),
        # channels of mixed visibility counts and image sizes as one graph
        dict(kind="batch", name="batch_ms2dirty", direction="ms2dirty", channels=12, low=16, high=21,
             eps=1e-5, mix=1),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _planes(c):
    """About how many w-planes an image case needs."""
    half = 0.5 * math.radians(c["fov"])
    r2 = min(0.99, half * half * (1.0 + (c["ny"] / c["nx"]) ** 2))
    wmax = {"tracks": c["extent"], "gauss": c["extent"] / 30.0,
            "uniform": 0.5 * c["nx"] / math.radians(c["fov"])}[c["coverage"]]
    kw = math.ceil(-math.log10(c["eps"] / 10.0))
    return 4.0 * (1.0 - math.sqrt(1.0 - r2)) * wmax + kw + 1


def draw(rng):
    kind = rng.choice(["image"] * 4 + ["nufft", "batch"])
    if kind == "nufft":
        double = rng.random() < 0.3
        return dict(kind="nufft", type=rng.choice(["1", "2"]), points=int(_log(rng, 2e3, 1.6e7)),
                    n1=int(_log(rng, 60, 2000 if double else 4096)), n2=int(_log(rng, 60, 2000 if double else 4096)),
                    eps=rng.choice([1e-7, 1e-10, 1e-12] if double else [1e-3, 1e-4, 1e-5, 1e-6]),
                    double=double, clustered=rng.random() < 0.5)
    if kind == "batch":
        low = rng.randint(13, 17)
        return dict(kind="batch", direction=rng.choice(["ms2dirty", "dirty2ms"]),
                    channels=rng.randint(4, 12), low=low, high=low + rng.randint(1, 4),
                    eps=rng.choice([1e-4, 1e-5]), mix=rng.randint(2, 1000))
    double = rng.random() < 0.3
    nx = int(_log(rng, 64, 2048 if double else 4096))
    ny = nx if rng.random() < 0.4 else min(4096, max(48, int(nx * _log(rng, 0.4, 2.0))))
    channels = rng.choice([1, 1, 1, 2, 5, 16])
    c = _image(None, rng.choice(["ms2dirty", "dirty2ms"]), int(_log(rng, 1e3, 4e6) / channels) + 2, nx, ny,
               rng.uniform(1.0, 10.0), 1e9 * rng.uniform(0.5, 1.6),
               rng.choice([1e-7, 1e-9, 1e-12] if double else [1e-3, 1e-4, 1e-5, 1e-6]),
               rng.choice(["tracks", "tracks", "gauss", "uniform"]), channels=channels, double=double,
               uvw32=(not double) and rng.random() < 0.2, weights=rng.random() < 0.6,
               wstacking=rng.random() < 0.85, shuffled=rng.random() < 0.3, host=rng.random() < 0.15)
    c["host"] = c["host"] and (double or channels > 1)
    if c["host"]:
        c["uvw32"] = False
        c["rows"] = min(c["rows"], 200000 // channels)
    # the coverage stays inside the grid (|u| pixel < 1/2) and the w-planes
    # inside about 16 GB
    cell = 16 if double else 8
    while True:
        c["extent"] = 0.2 * nx / math.radians(c["fov"]) / _log(rng, 1.0, 4.0)
        if 4.0 * c["nx"] * c["ny"] * _planes(c) * cell < 16e9 or c["fov"] < 0.2:
            return c
        c["fov"] *= 0.7


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _complex(g, shape, double):
    t = torch.float64 if double else torch.float32
    return torch.complex(torch.randn(shape, generator=g, device="cuda", dtype=t),
                         torch.randn(shape, generator=g, device="cuda", dtype=t))


def _tracks(g, rows, shuffled):
    """uvw [rows, 3] of Earth-rotation tracks (8 h toward declination 45 deg,
    latitude 45 deg) scaled so that the longest baseline is 1; in time order
    with the array's baselines inside each time, or drawn at random."""
    nant = 27 if rows < 1 << 16 else 64 if rows < 1 << 20 else 256
    r = torch.sqrt(_rand(g, nant))
    th = 2 * math.pi * _rand(g, nant)
    east, north = r * torch.cos(th), r * torch.sin(th)
    s45 = math.sqrt(0.5)
    pos = torch.stack([-s45 * north, east, s45 * north])
    ii, jj = torch.triu_indices(nant, nant, 1, device="cuda")
    base = pos[:, jj] - pos[:, ii]
    base = base / base.square().sum(0).max().sqrt()
    nb = base.shape[1]
    out = torch.empty(rows, 3, device="cuda", dtype=torch.float64)
    steps = max(1, (rows + nb - 1) // nb)
    block = 1 << 24
    for lo in range(0, rows, block):
        n = min(block, rows - lo)
        if shuffled:
            b = torch.randint(0, nb, (n,), generator=g, device="cuda")
            hour = (_rand(g, n) * 2 - 1) * (math.pi / 3)
            sgn = torch.randint(0, 2, (n,), generator=g, device="cuda").double() * 2 - 1
        else:
            j = torch.arange(lo, lo + n, device="cuda")
            b = j % nb
            hour = ((j // nb).double() + 0.5) * (2.0 * math.pi / 3 / steps) - math.pi / 3
            sgn = torch.ones(n, device="cuda", dtype=torch.float64)
        x, y, z = base[0, b] * sgn, base[1, b] * sgn, base[2, b] * sgn
        sh, ch = torch.sin(hour), torch.cos(hour)
        out[lo:lo + n, 0] = sh * x + ch * y
        out[lo:lo + n, 1] = -s45 * ch * x + s45 * sh * y + s45 * z
        out[lo:lo + n, 2] = s45 * ch * x - s45 * sh * y + s45 * z
    return out


def _freqs(c):
    """The channels' frequencies: the highest is freq (the coverage in
    wavelengths is given there), the band spans a tenth of it."""
    n = c["channels"]
    return np.array([c["freq"] * (1.0 - 0.1 * (n - 1 - k) / n) for k in range(n)])


def _uvw(c, g):
    """FP64 uvw in metres.  extent: tracks' longest baseline, and six standard
    deviations of the Gaussian u and v, in wavelengths."""
    lam, rows = C_LIGHT / c["freq"], c["rows"]
    if c["coverage"] == "tracks":
        return _tracks(g, rows, c["shuffled"]) * (c["extent"] * lam)
    if c["coverage"] == "gauss":
        uvw = torch.randn(rows, 3, generator=g, device="cuda", dtype=torch.float64).clamp_(-5.5, 5.5)
        uvw *= c["extent"] * lam / 6.0
        uvw[:, 2] = (_rand(g, rows) * 2 - 1) * (c["extent"] * lam / 30.0)
        return uvw
    span = 0.999 * lam * c["nx"] / math.radians(c["fov"])
    uvw = (_rand(g, rows, 3) - 0.5) * span
    uvw[:, 1] *= c["ny"] / c["nx"]
    return uvw


def _image_inputs(c, seed):
    g = _gen(seed)
    uvw = _uvw(c, g)
    if c["uvw32"]:
        uvw = uvw.float()
    n = (c["rows"],) if c["channels"] == 1 else (c["rows"], c["channels"])
    real = torch.float64 if c["double"] else torch.float32
    wgt = None
    if c["weights"]:
        wgt = torch.rand(n, generator=g, device="cuda", dtype=real) + 0.5
    if c["direction"] == "ms2dirty":
        return uvw, _complex(g, n, c["double"]), wgt
    img = torch.zeros(c["nx"], c["ny"], device="cuda", dtype=torch.complex128 if c["double"] else torch.complex64)
    img.real = torch.randn(c["nx"], c["ny"], generator=g, device="cuda", dtype=real)
    return uvw, img, wgt


def _nufft_inputs(c, seed):
    g = _gen(seed)
    m = c["points"]
    real = torch.float64 if c["double"] else torch.float32
    pts = torch.rand(m, 2, generator=g, device="cuda", dtype=real) * 2 - 1
    pts *= math.pi
    if c["clustered"]:  # four fifths in 16 Gaussian clusters
        nb = (4 * m) // 5
        means = (torch.rand(16, 2, generator=g, device="cuda", dtype=real) * 2 - 1) * math.pi
        pts[:nb] = means[torch.randint(0, 16, (nb,), generator=g, device="cuda")]
        pts[:nb] += 0.3 * torch.randn(nb, 2, generator=g, device="cuda", dtype=real)
        pts = torch.remainder(pts + math.pi, 2 * math.pi) - math.pi
    pts.clamp_(-3.1415925, 3.1415925)
    x, y = pts[:, 0].contiguous(), pts[:, 1].contiguous()
    data = {}
    if c["type"] != "2":
        data["c"] = _complex(g, (m,), c["double"])
    if c["type"] != "1":
        data["fk"] = _complex(g, (c["n2"], c["n1"]), c["double"])
    return x, y, data


def _batch_shapes(c):
    """(rows, image side, frequency) of every channel of a batch case."""
    r = random.Random(c["mix"])
    n = c["channels"]
    return [(int(2.0 ** r.uniform(c["low"], c["high"])), r.choice([512, 1024, 2048]),
             1.0e9 + 0.6e9 * k / max(1, n - 1)) for k in range(n)]


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "image":
        uvw, data, wgt = _image_inputs(c, seed)
        state = dict(case=c, freq=_freqs(c), uvw=uvw, data=data, wgt=wgt)
        if c["host"]:
            host = lambda t: None if t is None else t.cpu().numpy()  # noqa: E731
            state.update(uvw=host(uvw), data=host(data), wgt=host(wgt))
            if c["direction"] == "dirty2ms":
                state["data"] = np.ascontiguousarray(state["data"].real)
            return state
        state["ctx"] = _context()
        if c["direction"] == "ms2dirty":
            state["out"] = torch.empty(c["nx"], c["ny"], dtype=data.dtype, device="cuda")
        else:
            n = (c["rows"],) if c["channels"] == 1 else (c["rows"], c["channels"])
            state["out"] = torch.empty(n, dtype=data.dtype, device="cuda")
        return state
    if c["kind"] == "nufft":
        x, y, data = _nufft_inputs(c, seed)
        state = dict(case=c, ctx=_context(), x=x, y=y, **data)
        t = torch.complex128 if c["double"] else torch.complex64
        if c["type"] != "2":
            state["modes"] = torch.empty(c["n2"], c["n1"], dtype=t, device="cuda")
        if c["type"] != "1":
            state["points"] = torch.empty(c["points"], dtype=t, device="cuda")
        return state
    g = _gen(seed)
    items = []
    for rows, n, freq in _batch_shapes(c):
        # the full configuration's pixel size; baselines up to 7660
        # wavelengths at 1.4 GHz
        vis = _complex(g, (rows,), False)
        img = torch.zeros(n, n, device="cuda", dtype=torch.complex64)
        if c["direction"] == "dirty2ms":
            img.real = torch.randn(n, n, generator=g, device="cuda")
        items.append(dict(uvw=_tracks(g, rows, False) * (7660.0 * C_LIGHT / 1.4e9), vis=vis, wgt=None,
                          dirty=img, fov=3.0 / 8192 * n, freq=freq))
    out = [it["dirty" if c["direction"] == "ms2dirty" else "vis"] for it in items]
    return dict(case=c, batch=_context().batch(c["direction"], items, c["eps"]), out=out)


def run(state):
    c = state["case"]
    if c["kind"] == "image":
        if c["host"]:
            pix = math.radians(c["fov"]) / c["nx"]
            piy = math.radians(c["fov"]) / c["ny"]
            if c["direction"] == "ms2dirty":
                return cg.ms2dirty(state["uvw"], state["freq"], state["data"], state["wgt"], c["nx"], c["ny"],
                                   pix, piy, 0, 0, c["eps"], c["wstacking"])
            return cg.dirty2ms(state["uvw"], state["freq"], state["data"], state["wgt"], pix, piy, 0, 0,
                               c["eps"], c["wstacking"])
        ctx = state["ctx"]
        if c["direction"] == "ms2dirty":
            return ctx.ms2dirty(state["uvw"], state["data"], state["wgt"], c["nx"], c["ny"], c["fov"],
                                state["freq"], c["eps"], out=state["out"], do_wstacking=c["wstacking"])
        return ctx.dirty2ms(state["uvw"], state["data"], state["wgt"], c["fov"], state["freq"], c["eps"],
                            out=state["out"], do_wstacking=c["wstacking"])
    if c["kind"] == "nufft":
        ctx, out = state["ctx"], {}
        if c["type"] != "2":
            out["modes"] = ctx.nufft2d1(state["x"], state["y"], state["c"], c["n1"], c["n2"], c["eps"],
                                        out=state["modes"])
        if c["type"] != "1":
            out["points"] = ctx.nufft2d2(state["x"], state["y"], state["fk"], c["eps"], out=state["points"])
        return out
    state["batch"].run()
    return state["out"]


# ------------------------------------------------------------------ work

def _support(eps, double):
    return min(16, max(2, math.ceil(-math.log10(max(eps, 1.1e-16 if double else 6e-8) / 10.0))))


def _smooth(n):
    """Even grid side of at least 2n with no prime factor above 5."""
    m = 2 * n
    while True:
        k = m
        for p in (2, 3, 5):
            while k % p == 0:
                k //= p
        if k == 1:
            return m
        m += 2


def _work(points, rows, nx, ny, planes, eps, double, uvw_bytes, weights, axes):
    """Inputs and outputs moved once; spreading or interpolating every point
    (kw^axes taps, a complex multiply-add with a real factor each), the
    transforms of the planes, and the planes' phases on the image."""
    cell = 16 if double else 8
    kw = _support(eps, double)
    cells = float(_smooth(nx)) * _smooth(ny) * planes
    nbytes = rows * uvw_bytes + points * cell + (points * cell / 2 if weights else 0) + nx * ny * cell
    flops = points * 4.0 * kw ** axes + 5.0 * cells * math.log2(max(2.0, 4.0 * nx * ny)) + 8.0 * nx * ny * planes
    return {"bytes": float(nbytes), "flops": flops}


def work(case):
    c = case
    if c["kind"] == "image":
        planes = _planes(c) if c["wstacking"] else 1
        return _work(c["rows"] * c["channels"], c["rows"], c["nx"], c["ny"], planes, c["eps"], c["double"],
                     12 if c["uvw32"] else 24, c["weights"], 3 if c["wstacking"] else 2)
    if c["kind"] == "nufft":
        one = _work(c["points"], c["points"], c["n1"], c["n2"], 1, c["eps"], c["double"],
                    16 if c["double"] else 8, False, 2)
        times = 2 if c["type"] == "both" else 1
        return {k: v * times for k, v in one.items()}
    total = {"bytes": 0.0, "flops": 0.0}
    for rows, n, freq in _batch_shapes(c):
        p = _planes(dict(coverage="tracks", extent=7660.0 * freq / 1.4e9, nx=n, ny=n, fov=3.0 / 8192 * n, eps=c["eps"]))
        for k, v in _work(rows, rows, n, n, p, c["eps"], False, 24, False, 3).items():
            total[k] += v
    return total


# ------------------------------------------------------------------ exact

MOST_TERMS = 4.5e11  # point-pixel pairs of a direct sum: about 15 seconds


def _directions(c):
    """l, m and n - 1 of every pixel, FP64 [nx * ny] each (0 for n - 1 and
    without 1/n when w is ignored)."""
    px, py = math.radians(c["fov"]) / c["nx"], math.radians(c["fov"]) / c["ny"]
    l = (torch.arange(c["nx"], device="cuda", dtype=torch.float64) - c["nx"] // 2) * px
    m = (torch.arange(c["ny"], device="cuda", dtype=torch.float64) - c["ny"] // 2) * py
    l, m = l[:, None].expand(c["nx"], c["ny"]).reshape(-1), m[None, :].expand(c["nx"], c["ny"]).reshape(-1)
    r2 = l * l + m * m
    nm1 = -r2 / (torch.sqrt(torch.clamp(1.0 - r2, min=0.0)) + 1.0)
    return l, m, nm1 if c["wstacking"] else torch.zeros_like(nm1)


def _direct(turns_a, values, turns_b, block):
    """sum_j values[j] exp(2 pi i a_k . b_j) for every k: a [K, 3], b [J, 3],
    complex values [J]."""
    out = torch.empty(turns_a.shape[0], dtype=torch.complex128, device="cuda")
    bt = turns_b.t().contiguous()
    re, im = values.real.contiguous(), values.imag.contiguous()
    for lo in range(0, turns_a.shape[0], block):
        t = turns_a[lo:lo + block] @ bt
        t -= torch.round(t)
        t *= 2.0 * math.pi
        s, k = torch.sin(t), t.cos_()
        out[lo:lo + block] = torch.complex((k * re).sum(1) - (s * im).sum(1), (k * im).sum(1) + (s * re).sum(1))
    return out


def _exact_image(c, seed):
    points = c["rows"] * c["channels"]
    if float(points) * c["nx"] * c["ny"] > MOST_TERMS:
        return None
    uvw, data, wgt = _image_inputs(c, seed)
    f = torch.tensor(_freqs(c) / C_LIGHT, device="cuda")
    # w enters with sign -1, and turns of u l + v m + w (n - 1) per point
    b = uvw.double()[:, None, :] * f[None, :, None]
    b = (b * torch.tensor([1.0, 1.0, -1.0], device="cuda", dtype=torch.float64)).reshape(-1, 3)
    l, m, nm1 = _directions(c)
    a = torch.stack([l, m, nm1], 1)
    w = None if wgt is None else wgt.double().reshape(-1)
    if c["direction"] == "ms2dirty":
        v = data.to(torch.complex128).reshape(-1)
        img = _direct(a, v if w is None else v * w, b, max(1, (1 << 27) // points))
        img = (img / (nm1 + 1.0)).reshape(c["nx"], c["ny"])
        return img.real.cpu().numpy() if c["host"] else img
    d = (data.to(torch.complex128).reshape(-1) / (nm1 + 1.0))
    vis = _direct(-b, d, a, max(1, (1 << 27) // (c["nx"] * c["ny"])))
    vis = vis if w is None else vis * w
    if c["host"]:
        return vis.reshape(c["rows"], c["channels"]).cpu().numpy()
    return vis if c["channels"] == 1 else vis.reshape(c["rows"], c["channels"])


def _exact_nufft(c, seed):
    if float(c["points"]) * c["n1"] * c["n2"] > 2e13:
        return None
    x, y, data = _nufft_inputs(c, seed)
    out = {}
    k1 = torch.arange(c["n1"], device="cuda", dtype=torch.float64) - c["n1"] // 2
    k2 = torch.arange(c["n2"], device="cuda", dtype=torch.float64) - c["n2"] // 2
    block = max(1, (1 << 26) // (c["n1"] + c["n2"]))
    modes = torch.zeros(c["n2"], c["n1"], dtype=torch.complex128, device="cuda")
    pts = torch.empty(c["points"], dtype=torch.complex128, device="cuda")
    for lo in range(0, c["points"], block):
        xs, ys = x[lo:lo + block].double(), y[lo:lo + block].double()
        e1 = torch.polar(torch.ones((), device="cuda", dtype=torch.float64).expand(xs.numel(), c["n1"]), xs[:, None] * k1)
        e2 = torch.polar(torch.ones((), device="cuda", dtype=torch.float64).expand(c["n2"], xs.numel()), k2[:, None] * ys)
        if c["type"] != "2":
            modes += e2 @ (data["c"][lo:lo + block].to(torch.complex128)[:, None] * e1)
        if c["type"] != "1":
            t = e2.conj().resolve_conj().t().contiguous() @ data["fk"].to(torch.complex128)
            pts[lo:lo + block] = (t * e1.conj()).sum(1)
    if c["type"] != "2":
        out["modes"] = modes
    if c["type"] != "1":
        out["points"] = pts
    return out


def exact(case, seed):
    c = dict(case)
    if c["kind"] == "image":
        return _exact_image(c, seed)
    if c["kind"] == "nufft":
        return _exact_nufft(c, seed)
    return None
