"""Performance cases: the work that users of this package have it do, over its real range.

`listed()` names the standing cases, `draw(rng)` makes more of the same ranges, `prepare`
builds what a program holds before the call (inputs on the GPU and any plan it keeps),
`run` makes one pass through the public entry points, `work` counts the bytes and
operations the pass cannot do without, and `exact` gives the same outputs in 64 bits from
plain torch.

Kinds of case:
  das      one delay-and-sum problem: forward, forward + adjoint called by hand, or through
           autograd; dense or sparse compounding; linear or matrix probe
  batched  das_batched over the three mixed probes (sparse compounding of frame ensembles)
  rank     the clutter filter, truncate_rank
  interp   scan conversion: evaluation with a kept plan, or the one-shot call
  greens   frequency-domain simulation

Units: positions in sampling wavelengths (c / fs), delays in samples, as the package's.
"""
import math

import torch

import ffdas_amd

C_SOUND = 1540.0
FS = 40e6
F0 = 5e6
KS = FS / C_SOUND          # sampling wavelengths per metre
RADIUS_SQ_MIN = 1.0000000116860974e-07   # the FP32 value of 1e-7


# ------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------
def das_case(name=None, probe="linear", channels=128, tx=3, samples=2048, frames=1, nz=256,
             ny=1, nx=128, data="f32", mode="forward", sparse=0, directivity=False,
             scale=1.0, trailing=False):
    c = dict(kind="das", probe=probe, channels=channels, tx=tx, samples=samples, frames=frames,
             nz=nz, ny=ny, nx=nx, data=data, mode=mode, sparse=sparse, directivity=directivity,
             scale=scale, trailing=trailing)
    return c if name is None else dict(c, name=name)


def batched_case(name=None, frames=16, tx=64, samples=2048, sparse=8, linear=128, wide=192,
                 cube=64):
    c = dict(kind="batched", frames=frames, tx=tx, samples=samples, sparse=sparse,
             linear=linear, wide=wide, cube=cube)
    return c if name is None else dict(c, name=name)


def rank_case(name=None, frames=64, voxels=64 ** 3, dtype="c64", start=5, stop=0):
    c = dict(kind="rank", frames=frames, voxels=voxels, dtype=dtype, start=start, stop=stop)
    return c if name is None else dict(c, name=name)


def interp_case(name=None, frames=16, nr=512, nt=96, nphi=96, query=256, dtype="f32",
                planned=True, nearest=False):
    c = dict(kind="interp", frames=frames, nr=nr, nt=nt, nphi=nphi, query=query, dtype=dtype,
             planned=planned, nearest=nearest)
    return c if name is None else dict(c, name=name)


def greens_case(name=None, events=8, sources=128, freqs=512, nz=256, nx=128):
    c = dict(kind="greens", events=events, sources=sources, freqs=freqs, nz=nz, nx=nx)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # a live preview: one plane wave, one frame, a coarse image; host time and launches count
        das_case("das_preview", channels=64, tx=1, samples=1024, nz=64, nx=64),
        # plain 2-D beamforming of one frame, three plane waves (the package's first workload)
        das_case("das_plane_2d", channels=128, tx=3, samples=2048, nz=256, nx=128),
        # demodulated data in half2, a short ensemble
        das_case("das_iq_half2", channels=128, tx=3, samples=2048, frames=8, nz=256, nx=128,
                 data="c16"),
        # one volume of a 32 x 32 matrix probe: the largest single forward call
        das_case("das_volume", probe="matrix", channels=1024, tx=16, samples=4096, nz=128,
                 ny=128, nx=128, directivity=True),
        # differentiable beamforming, the headline workload: FP16 data, 16 frames, forward and
        # adjoint called by hand as a training loop that owns its step does
        das_case("das_step_fp16", channels=128, tx=11, samples=2048, frames=16, nz=256, nx=256,
                 data="f16", mode="step"),
        # the same through autograd in FP32 on a small batch of ragged size, gradients of the
        # data, the delays and the apodization
        das_case("das_autograd_fp32", channels=96, tx=5, samples=1500, frames=6, nz=201, nx=151,
                 mode="autograd", scale=1.02),
        # sparse compounding of frame ensembles from mixed probes in one call
        batched_case("das_sparse_mixed"),
        # clutter filter of a 64-frame complex ensemble
        rank_case("rank_clutter_c64"),
        # clutter filter of a long real ensemble
        rank_case("rank_long_f32", frames=200, voxels=96 ** 3, dtype="f32", start=3),
        # scan conversion of an ensemble with the plan and the point location kept
        interp_case("interp_ensemble"),
        # one-shot scan conversion of one volume: plan, location and evaluation in one call
        interp_case("interp_oneshot", frames=1, nr=256, nt=64, nphi=64, query=128, planned=False),
        # array simulation, eight transmit events
        greens_case("greens_events8"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_das(rng):
    matrix = rng.random() < 0.3
    mode = rng.choice(["forward", "forward", "step", "autograd"])
    data = rng.choice(["f32", "f32", "f16", "bf16", "f32to16", "c32", "c16"]
                      if mode == "forward" else ["f32", "f16", "bf16"])
    if matrix:
        side = rng.randint(8, 32)
        c = das_case(probe="matrix", channels=side * side, tx=_log_int(rng, 1, 16),
                     samples=rng.randint(700, 4096), frames=rng.choice([1, 1, 2, 4, 8]),
                     nz=_log_int(rng, 16, 96), ny=_log_int(rng, 12, 96), nx=_log_int(rng, 12, 96),
                     data=data, mode=mode, directivity=rng.random() < 0.5)
    else:
        c = das_case(channels=rng.choice([32, 64, 96, 128, 128, 192, 256, rng.randint(17, 256)]),
                     tx=_log_int(rng, 1, 32), samples=rng.randint(512, 4096),
                     frames=rng.choice([1, 1, 2, 4, 6, 8, 16, 16, 20, 32]),
                     nz=_log_int(rng, 48, 400), nx=_log_int(rng, 48, 300), data=data, mode=mode)
    if rng.random() < 0.25:
        c["tx"] = max(c["tx"], 9)
        c["sparse"] = rng.choice([4, 8, 8, rng.randint(1, 9)])
    c["trailing"] = rng.random() < 0.15
    if mode != "forward":
        c["scale"] = rng.choice([1.0, 1.0, round(rng.uniform(0.95, 1.05), 3)])
    most = 1.5e10 if mode == "forward" else 2.5e9
    cells = 3.0e8                             # samples of channel data
    while _units(c) > most or c["channels"] * c["tx"] * c["samples"] * c["frames"] > cells:
        big = max(("frames", "nz", "ny", "nx"), key=lambda k: c[k])
        if c["channels"] * c["tx"] * c["samples"] * c["frames"] > cells:
            big = "frames" if c["frames"] > 1 else "samples"
        c[big] = max(1, c[big] * 2 // 3)
    return c


def draw(rng):
    u = rng.random()
    if u < 0.46:
        return _draw_das(rng)
    if u < 0.54:
        return batched_case(frames=rng.choice([4, 8, 12, 16]), tx=rng.randint(16, 64),
                            samples=rng.randint(1024, 2048), sparse=rng.choice([4, 8]),
                            linear=rng.randint(48, 128), wide=rng.randint(64, 192),
                            cube=rng.randint(20, 64))
    if u < 0.70:
        dtype = rng.choice(["f32", "c64", "c64", "f64"])
        frames = _log_int(rng, 8, 60 if dtype == "f64" else 200)
        start = rng.randint(1, max(1, frames // 10))
        stop = rng.choice([0, 0, min(frames, start + rng.randint(1, max(1, frames // 4)))])
        return rank_case(frames=frames, voxels=_log_int(rng, 4000, 2 ** 27 // frames), dtype=dtype,
                         start=start, stop=stop)
    if u < 0.84:
        planned = rng.random() < 0.6
        return interp_case(frames=rng.choice([1, 2, 4, 8, 11, 16, 32]) if planned else 1,
                           nr=_log_int(rng, 64, 400), nt=_log_int(rng, 16, 90),
                           nphi=_log_int(rng, 16, 90), query=_log_int(rng, 40, 180),
                           dtype=rng.choice(["f32", "f32", "c64"]), planned=planned,
                           nearest=rng.random() < 0.2)
    return greens_case(events=rng.choice([1, 1, 2, 3, 4, 6, 8, 11, 16]),
                       sources=rng.choice([32, 64, 128, rng.randint(20, 192)]),
                       freqs=_log_int(rng, 16, 512), nz=_log_int(rng, 32, 256),
                       nx=_log_int(rng, 24, 128))


# ------------------------------------------------------------------------------------------
# geometry and data
# ------------------------------------------------------------------------------------------
def _dev():
    return torch.device("cuda:0")


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed) * 7919 + 17)


def _span(n, half):
    return torch.linspace(-half, half, n, dtype=torch.float64, device=_dev()) if n > 1 else \
        torch.zeros(1, dtype=torch.float64, device=_dev())


def _elements(probe, channels, pitch=0.3e-3):
    if probe == "linear":
        x = (torch.arange(channels, dtype=torch.float64, device=_dev()) - (channels - 1) / 2) * pitch
        return torch.stack([x, torch.zeros_like(x), torch.zeros_like(x)], -1)
    side = int(round(math.sqrt(channels)))
    e = (torch.arange(side, dtype=torch.float64, device=_dev()) - (side - 1) / 2) * pitch
    ex, ey = torch.meshgrid(e, e, indexing="ij")
    return torch.stack([ex.reshape(-1), ey.reshape(-1), torch.zeros(side * side, device=_dev(),
                                                                    dtype=torch.float64)], -1)


def _units(c):
    slots = c["sparse"] or c["tx"]
    return c["nz"] * c["ny"] * c["nx"] * c["channels"] * slots * c["frames"]


def _traces(shape, samples, dtype, g):
    """Speckle-like channel data: every row a stretch of band-passed (complex: low-passed)
    Gaussian noise of unit variance, plus a little white noise's worth of independence from
    its random start."""
    n = 1 << 20
    f = torch.fft.rfftfreq(n, device=_dev(), dtype=torch.float32)
    if dtype.is_complex:
        f = torch.fft.fftfreq(n, device=_dev(), dtype=torch.float32)
        band = torch.exp(-0.5 * (f / 0.03) ** 2)
        z = torch.complex(torch.randn(n, device=_dev(), generator=g),
                          torch.randn(n, device=_dev(), generator=g))
        bank = torch.fft.ifft(torch.fft.fft(z) * band)
    else:
        band = torch.exp(-0.5 * ((f - F0 / FS) / 0.03) ** 2)
        bank = torch.fft.irfft(torch.fft.rfft(torch.randn(n, device=_dev(), generator=g)) * band, n)
    bank = bank / bank.abs().square().mean().sqrt()
    if not dtype.is_complex:
        bank = bank.to(dtype)
    rows = math.prod(shape)
    start = torch.randint(0, n - samples, (rows,), device=_dev(), generator=g)
    out = torch.empty((rows, samples), dtype=bank.dtype, device=_dev())
    stretch = bank.unfold(0, samples, 1)
    step = max(1, (1 << 27) // samples)
    for a in range(0, rows, step):
        out[a:a + step] = stretch[start[a:a + step]]
    return out.reshape(tuple(shape) + (samples,))


def _focused(points, foci):
    d = torch.linalg.vector_norm(points[None] - foci.reshape((-1,) + (1,) * (points.ndim - 1) + (3,)),
                                 dim=-1)
    z = foci[:, 2].reshape((-1,) + (1,) * (points.ndim - 1))
    sign = torch.where(points[None, ..., 2] >= z, 1.0, -1.0)
    return (z + sign * d) * KS


def _nearest(points, foci, k):
    """int32 (k, *points): the k foci of least lateral distance, in chunks of points."""
    flat = points.reshape(-1, 3)
    idx = torch.empty((flat.shape[0], k), dtype=torch.int32, device=_dev())
    for a in range(0, flat.shape[0], 1 << 18):
        d = torch.linalg.vector_norm(flat[a:a + (1 << 18), None, :2] - foci[None, :, :2], dim=-1)
        idx[a:a + (1 << 18)] = torch.sort(d, dim=-1, stable=True).indices[:, :k].to(torch.int32)
    return idx.t().contiguous().reshape((k,) + tuple(points.shape[:-1]))


def _geometry(probe, channels, tx, sparse, nz, ny, nx, directivity, samples, scale=1.0):
    """Element and voxel positions, delays, weights and tables of one problem."""
    matrix = probe == "matrix"
    elem = _elements(probe, channels)
    # the depth whose round trip still fits the record, less the aperture's own spread
    deepest = 0.5 * samples / KS - 2e-3
    z0, z1 = (5e-3, max(8e-3, min(50e-3 if matrix else 45e-3, deepest)))
    z = torch.linspace(z0, z1, nz, dtype=torch.float64, device=_dev())
    half = float(elem[:, 0].abs().max())
    if matrix:
        lat = max(half, 15e-3 if directivity else 9.6e-3)
        zz, yy, xx = torch.meshgrid(z, _span(ny, lat), _span(nx, lat), indexing="ij")
        grid = torch.stack([xx, yy, zz], -1)
    else:
        zz, xx = torch.meshgrid(z, _span(nx, half), indexing="ij")
        grid = torch.stack([xx, torch.zeros_like(xx), zz], -1)
    table = None
    if sparse:
        if matrix:
            m = max(1, int(round(math.sqrt(tx))))
            gx, gy = torch.meshgrid(_span(m, 9.6e-3), _span(m, 9.6e-3), indexing="ij")
            foci = torch.stack([gx.reshape(-1), gy.reshape(-1),
                                torch.full((m * m,), 0.5 * (z0 + z1), device=_dev(),
                                           dtype=torch.float64)], -1)[:tx]
        else:
            fx = _span(tx, half)
            foci = torch.stack([fx, torch.zeros_like(fx), torch.full_like(fx, 0.5 * (z0 + z1))], -1)
        sparse = min(sparse, foci.shape[0])
        table = _nearest(grid, foci, sparse)
        offs = torch.gather(_focused(grid, foci), 0, table.long())
        weights = torch.full(offs.shape, 1.0 / sparse, device=_dev())
    elif matrix:
        m = max(1, int(math.ceil(math.sqrt(tx))))
        e = (torch.arange(m, dtype=torch.float64, device=_dev()) - (m - 1) / 2) * 3e-3
        vx, vy = torch.meshgrid(e, e, indexing="ij")
        src = torch.stack([vx.reshape(-1), vy.reshape(-1),
                           torch.full((m * m,), -10e-3, device=_dev(), dtype=torch.float64)], -1)[:tx]
        over = (src[:, :2].abs() - half).clamp(min=0)
        ref = (over.square().sum(-1) + src[:, 2].square()).sqrt()
        vec = grid[None] - src.reshape(-1, 1, 1, 1, 3)
        dist = torch.linalg.vector_norm(vec, dim=-1)
        offs = (dist - ref.reshape(-1, 1, 1, 1)) * KS
        ratio = torch.tan(torch.acos((vec[..., 2] / dist).clamp(-1, 1)))
        weights = torch.where(ratio.abs() <= 0.5, 0.5 + 0.5 * torch.cos(2 * math.pi * ratio),
                              torch.zeros_like(ratio))
    else:
        th = torch.deg2rad(_span(tx, 15.0)).reshape(-1, 1, 1)
        offs = (grid[..., 2] * torch.cos(th) + grid[..., 0] * torch.sin(th)) * KS
        weights = torch.full(offs.shape, 1.0 / tx, device=_dev())
    srcdir = None
    if directivity:
        srcdir = torch.tensor([0.0, 0.0, 1.0, math.cos(math.radians(30.0))], device=_dev())
        srcdir = srcdir.expand(elem.shape[0], 4).contiguous()
    f = lambda t: t.to(torch.float32).contiguous()
    return dict(srcpos=f(elem * KS), dstpos=f(grid * KS), offsets=f(offs), weights=f(weights),
                srcdir=srcdir, table=table)


_STORE = {"f32": torch.float32, "f32to16": torch.float32, "f16": torch.float16,
          "bf16": torch.bfloat16, "c32": torch.complex64, "c16": torch.complex64}


def _das_inputs(case, seed):
    g = _gen(seed)
    geo = _geometry(case["probe"], case["channels"], case["tx"], case["sparse"], case["nz"],
                    case["ny"], case["nx"], case["directivity"], case["samples"])
    C, T = geo["srcpos"].shape[0], case["tx"]
    shape = (case["frames"],) + ((T, C) if case["trailing"] else (C, T))
    x = _traces(shape, case["samples"], _STORE[case["data"]], g)
    if case["data"] == "c16":
        x = torch.view_as_real(x).half()
    spatial = tuple(geo["dstpos"].shape[:-1])
    target = torch.randn((case["frames"],) + spatial, device=_dev(), generator=g)
    return geo, x, target


def _sector(nr, nt, nphi, dtype=torch.float64):
    """Vertices of a volumetric sector scan: radius and two steering angles."""
    r = torch.linspace(0.05, 1.0, nr, dtype=torch.float64, device=_dev())
    th, ph = _span(nt, 0.6), _span(nphi, 0.6)
    R, TH, PH = torch.meshgrid(r, th, ph, indexing="ij")
    return torch.stack([R * torch.sin(TH) * torch.cos(PH), R * torch.sin(PH),
                        R * torch.cos(TH) * torch.cos(PH)], -1).to(dtype)


def _interp_inputs(case, seed):
    g = _gen(seed)
    grid = _sector(case["nr"], case["nt"], case["nphi"], torch.float32)
    lo, hi = grid.reshape(-1, 3).amin(0), grid.reshape(-1, 3).amax(0)
    # a Cartesian raster over the sector's box, shifted by part of a step: another view of it
    n = case["query"]
    shift = torch.rand(3, device=_dev(), generator=g) * 0.5
    ax = [lo[k] + (hi[k] - lo[k]) * (torch.arange(n, device=_dev()) + shift[k]) / n for k in range(3)]
    Z, Y, X = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    q = torch.stack([X, Y, Z], -1).contiguous()
    shape = (case["frames"], case["nr"], case["nt"], case["nphi"])
    x = torch.randn(shape, device=_dev(), generator=g)
    if case["dtype"] == "c64":
        x = torch.complex(x, torch.randn(shape, device=_dev(), generator=g))
    return grid, q, x


def _rank_inputs(case, seed):
    """Tissue in the first `start` components (18 to 22 dB above the noise each), a weaker flow in
    the kept ones where the case keeps a band, noise in all."""
    g = _gen(seed)
    m, n = case["frames"], case["voxels"]
    base = torch.float64 if case["dtype"] == "f64" else torch.float32
    cplx = case["dtype"] == "c64"

    def normal(*s):
        v = torch.randn(s, device=_dev(), generator=g, dtype=base)
        return torch.complex(v, torch.randn(s, device=_dev(), generator=g, dtype=base)) if cplx else v

    x = normal(m, n)
    k = case["stop"] or case["start"]
    u = torch.linalg.qr(normal(m, m).cpu()).Q.to(_dev())[:, :k] * math.sqrt(m)
    amp = torch.full((k,), 3.0, device=_dev(), dtype=base)
    tissue = torch.arange(case["start"], device=_dev(), dtype=base)
    amp[:case["start"]] = 12.0 - 4.0 * tissue / max(1, case["start"])
    return x.addmm_(u * amp, normal(k, n))


def _greens_inputs(case, seed):
    g = _gen(seed)
    ns, nf = case["sources"], case["freqs"]
    src = torch.zeros((ns, 3), device=_dev(), dtype=torch.float64)
    src[:, 0] = (torch.arange(ns, device=_dev()) - (ns - 1) / 2) * 0.3e-3
    zz, xx = torch.meshgrid(torch.linspace(5e-3, 45e-3, case["nz"], device=_dev(), dtype=torch.float64),
                            _span(case["nx"], 19e-3), indexing="ij")
    dst = torch.stack([xx, torch.zeros_like(xx), zz], -1)
    f = F0 + (torch.arange(nf, device=_dev(), dtype=torch.float64) - nf / 2) * (8e6 / nf)
    shape = (case["events"], ns, nf)
    x = torch.complex(torch.randn(shape, device=_dev(), generator=g),
                      torch.randn(shape, device=_dev(), generator=g))
    return src.float(), (-2 * math.pi * f / C_SOUND).float(), x, dst.float()


_PROBES = (("linear", 64, "linear"), ("linear", 256, "wide"), ("matrix", 1024, "cube"))


def _batched_inputs(case, seed):
    g = _gen(seed)
    problems = []
    for probe, channels, key in _PROBES:
        n = case[key]
        geo = _geometry(probe, channels, case["tx"], case["sparse"], n, n if probe == "matrix" else 1,
                        n, False, case["samples"])
        x = _traces((case["frames"], channels, case["tx"]), case["samples"], torch.float16, g)
        problems.append(dict(x=x, srcpos=geo["srcpos"], dstpos=geo["dstpos"], offsets=geo["offsets"],
                             weights=geo["weights"], sparse_indices=geo["table"]))
    return problems


# ------------------------------------------------------------------------------------------
# a pass
# ------------------------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "das":
        geo, x, target = _das_inputs(case, seed)
        s = dict(geo, case=case, x=x)
        if case["data"] == "c16":
            s["x"] = ffdas_amd.view(x, ffdas_amd.half2)
        s["wavenum"] = 2 * math.pi * F0 / FS if case["data"][0] == "c" else 0.0
        if case["mode"] == "step":
            s["neg2_target"] = -2.0 * target
        elif case["mode"] == "autograd":
            s["grad_out"] = target
            for k in ("x", "offsets", "weights"):
                s[k].requires_grad_(True)
        return s
    if case["kind"] == "batched":
        return dict(case=case, problems=_batched_inputs(case, seed))
    if case["kind"] == "rank":
        x = _rank_inputs(case, seed)
        return dict(case=case, x=x, out=torch.empty_like(x))
    if case["kind"] == "interp":
        grid, q, x = _interp_inputs(case, seed)
        s = dict(case=case, grid=grid, q=q, x=x, mode="nearest" if case["nearest"] else "linear")
        if case["planned"]:
            s["plan"] = ffdas_amd.Interpolator(grid, mode=s["mode"])
            s["plan"].preprocess(q)
            s["out"] = torch.empty((case["frames"],) + tuple(q.shape[:-1]), dtype=x.dtype,
                                   device=x.device)
        return s
    src, k, x, dst = _greens_inputs(case, seed)
    out = torch.empty((case["events"],) + tuple(dst.shape[:-1]) + (case["freqs"],),
                      dtype=torch.complex64, device=x.device)
    return dict(case=case, src=src, k=k, x=x, dst=dst, out=out)


def _forward(s):
    c = s["case"]
    more = dict(srcdir=s["srcdir"], wavenum=s["wavenum"], channels_trailing=c["trailing"],
                use_fp16=c["data"] == "f32to16", scale=c["scale"])
    geo = (s["srcpos"], s["dstpos"], s["offsets"], s["weights"])
    if s["table"] is not None:
        return ffdas_amd.das_sparse(s["x"], *geo, s["table"], **more)
    return ffdas_amd.das(s["x"], *geo, **more)


def run(state):
    c = state["case"]
    if c["kind"] == "das":
        out = _forward(state)
        if c["mode"] == "forward":
            return out
        if c["mode"] == "autograd":
            grads = torch.autograd.grad(out, (state["x"], state["offsets"], state["weights"]),
                                        state["grad_out"])
            return [out, *grads]
        # the gradient of sum (out - target)^2, then the adjoint on the unchanged data
        g = torch.add(state["neg2_target"], out, alpha=2.0)
        gx, go, _, gs = ffdas_amd.das_backward(
            state["x"], state["srcpos"], state["dstpos"], state["offsets"], state["weights"], g,
            srcdir=state["srcdir"], sparse_indices=state["table"], scale=c["scale"],
            channels_trailing=c["trailing"], need_weights=False, reuse_x=True)
        return [out, gx, go, gs]
    if c["kind"] == "batched":
        return ffdas_amd.das_batched(state["problems"])
    if c["kind"] == "rank":
        return ffdas_amd.truncate_rank(state["x"], c["start"], c["stop"] or None, out=state["out"])
    if c["kind"] == "interp":
        if c["planned"]:
            return state["plan"](state["x"], state["q"], out=state["out"])
        return ffdas_amd.interpolate(state["grid"], state["x"], state["q"], mode=state["mode"])
    return ffdas_amd.greens(state["src"], state["k"], state["x"], state["dst"], out=state["out"])


# ------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------
def _das_work(c):
    cplx = c["data"][0] == "c"
    size = {"f32": 4, "f32to16": 4, "f16": 2, "bf16": 2, "c32": 8, "c16": 4}[c["data"]]
    n = c["nz"] * c["ny"] * c["nx"]
    slots = c["sparse"] or c["tx"]
    x = c["frames"] * c["channels"] * c["tx"] * c["samples"]
    out = c["frames"] * n * (8 if cplx else 4)
    b = x * size + n * (12 + slots * (12 if c["sparse"] else 8)) + c["channels"] * 28 + out
    # per unit: two multiply-adds (complex: eight more for the rotated weight); per voxel,
    # channel and slot about ten for the delay
    flops = _units(c) * (12 if cplx else 4) + _units(c) // c["frames"] * 10
    if c["mode"] != "forward":
        b += out + x * 4 + n * slots * 4 * (2 if c["mode"] == "autograd" else 1)
        flops += _units(c) * 8 + _units(c) // c["frames"] * 10
    return b, flops


def work(case):
    k = case["kind"]
    if k == "das":
        b, f = _das_work(case)
    elif k == "batched":
        b = f = 0
        for probe, channels, key in _PROBES:
            n = case[key]
            sub = _das_work(dict(das_case(), channels=channels, tx=case["tx"], sparse=case["sparse"],
                                 samples=case["samples"], frames=case["frames"], data="f16",
                                 nz=n, ny=n if probe == "matrix" else 1, nx=n))
            b, f = b + sub[0], f + sub[1]
    elif k == "rank":
        m, n = case["frames"], case["voxels"]
        size = 4 if case["dtype"] == "f32" else 8
        cplx = 4 if case["dtype"] == "c64" else 1
        p, q = min(m, n), max(m, n)
        kept = (case["stop"] or p) - case["start"]
        r = min(kept, p - kept)
        b = 2 * m * n * size
        f = cplx * (p * (p + 1) * q + 4 * p * r * q + 4 * p ** 3 // 3)
    elif k == "interp":
        size = 8 if case["dtype"] == "c64" else 4
        nv, nq, B = case["nr"] * case["nt"] * case["nphi"], case["query"] ** 3, case["frames"]
        # a plan holds four vertex numbers and weights (nearest: one number) for each point
        lookup = nq * (4 if case["nearest"] else 32)
        b = B * (nv + nq) * size + (lookup if case["planned"] else nv * 12 + nq * 12)
        f = B * nq * 8 * (size // 4)
    else:
        nt = case["nz"] * case["nx"]
        b = case["events"] * case["freqs"] * 8 * (case["sources"] + nt) + nt * 12
        f = nt * case["sources"] * case["freqs"] * (8 * case["events"] + 10)
    return {"bytes": float(b), "flops": float(f)}


# ------------------------------------------------------------------------------------------
# the same outputs in 64 bits
# ------------------------------------------------------------------------------------------
def _das_exact(x, geo, *, wavenum=0.0, scale=1.0, grad_out=None):
    """x (B, C, T, S) in storage type -> out (B, *spatial) and, where grad_out(out) is given,
    the gradients (x, offsets, weights, scale) of real data; channel by channel."""
    B, C, T, S = x.shape
    spatial = tuple(geo["dstpos"].shape[:-1])
    dst = geo["dstpos"].detach().double().reshape(-1, 3)
    src = geo["srcpos"].double()
    N = dst.shape[0]
    ofs = geo["offsets"].detach().double().reshape(-1, N)
    w = geo["weights"].detach().double().reshape(-1, N)
    K = ofs.shape[0]
    tab = geo["table"].long().reshape(K, N) if geo["table"] is not None else None
    cplx = x.is_complex()
    wide = torch.complex128 if cplx else torch.float64
    wavenum = float(torch.tensor(wavenum, dtype=torch.float32))
    scale = float(torch.tensor(scale, dtype=torch.float32))

    def taps(c, k):
        d = dst - src[c]
        r = d.square().sum(-1).clamp(min=RADIUS_SQ_MIN).sqrt()
        tau = scale * (ofs[k] + r)
        kf = tau.floor()
        ok = (kf >= 0) & (kf < S - 1)
        if geo["srcdir"] is not None:
            sd = geo["srcdir"][c].double()
            ok = ok & ((d @ sd[:3]) / r > sd[3])
        row = tab[k] if tab is not None else torch.full_like(kf, k, dtype=torch.long)
        i = row * S + torch.where(ok, kf, torch.zeros_like(kf)).long()
        return r, tau, tau - kf, ok, i

    out = torch.zeros((B, N), dtype=wide, device=_dev())
    for c in range(C):
        data = x[:, c].reshape(B, T * S).to(wide)
        for k in range(K):
            _, tau, t, ok, i = taps(c, k)
            coef = torch.where(ok, w[k], torch.zeros_like(t))
            if cplx and wavenum:
                coef = torch.polar(coef, wavenum * tau)
            out.addcmul_(data[:, i], coef * (1 - t)).addcmul_(data[:, i + 1], coef * t)
    if grad_out is None:
        return out.reshape((B,) + spatial)
    g = grad_out(out.reshape((B,) + spatial)).double().reshape(B, N)
    gx = torch.zeros((B, C, T, S), dtype=torch.float64, device=_dev())
    go, gw = torch.zeros_like(ofs), torch.zeros_like(w)
    gs = torch.zeros((), dtype=torch.float64, device=_dev())
    for c in range(C):
        data = x[:, c].reshape(B, T * S).double()
        acc = torch.zeros((B, T * S), dtype=torch.float64, device=_dev())
        for k in range(K):
            r, _, t, ok, i = taps(c, k)
            coef = torch.where(ok, w[k], torch.zeros_like(t))
            v = coef * g
            acc.index_add_(1, i, v * (1 - t))
            acc.index_add_(1, i + 1, v * t)
            x0, x1 = data[:, i], data[:, i + 1]
            step = (g * (x1 - x0)).sum(0) * ok
            go[k] += scale * w[k] * step
            gw[k] += (g * (x0 + t * (x1 - x0))).sum(0) * ok
            gs += (w[k] * step * (ofs[k] + r)).sum()
        gx[:, c] = acc.reshape(B, T, S)
    return (out.reshape((B,) + spatial), gx, go.reshape((K,) + spatial),
            gw.reshape((K,) + spatial), gs)


def _natural(case, x):
    if case["data"] == "c16":
        x = torch.view_as_complex(x.float())
    return x.transpose(1, 2) if case["trailing"] else x


_TETS = ((0, 1, 2, 4), (1, 3, 2, 7), (1, 2, 4, 7), (2, 4, 6, 7), (1, 4, 5, 7))


def _interp_exact(case, grid, q, x):
    """Every grid cell is five tetrahedra (corners numbered with bit 0 for +x, bit 1 for +y, bit 2
    for +z); a point takes the weights of the first tetrahedron, by number, that holds it."""
    nr, nt, nphi = case["nr"], case["nt"], case["nphi"]
    v = grid.double().reshape(-1, 3)
    p = q.double().reshape(-1, 3)
    nq = p.shape[0]
    r = torch.linalg.vector_norm(p, dim=-1)
    place = torch.stack([(r - 0.05) / 0.95 * (nr - 1),
                         (torch.atan2(p[:, 0], p[:, 2]) / 1.2 + 0.5) * (nt - 1),
                         (torch.asin((p[:, 1] / r).clamp(-1, 1)) / 1.2 + 0.5) * (nphi - 1)], -1)
    cell0 = place.floor().long()
    top = torch.tensor([nr - 2, nt - 2, nphi - 2], device=_dev())
    near = ((cell0 >= -2) & (cell0 <= top + 2)).all(-1).nonzero()[:, 0]
    best = torch.full((nq,), 1 << 62, dtype=torch.long, device=_dev())
    ids = torch.zeros((nq, 4), dtype=torch.long, device=_dev())
    wts = torch.zeros((nq, 4), dtype=torch.float64, device=_dev())
    for shift in torch.cartesian_prod(*(torch.tensor([-1, 0, 1]),) * 3).tolist():
        cell = cell0[near] + torch.tensor(shift, device=_dev())
        inside = ((cell >= 0) & (cell <= top)).all(-1)
        at, cell = near[inside], cell[inside]
        base = (cell[:, 0] * nt + cell[:, 1]) * nphi + cell[:, 2]
        number = ((cell[:, 0] * (nt - 1) + cell[:, 1]) * (nphi - 1) + cell[:, 2]) * 6
        for j, tet in enumerate(_TETS):
            vid = torch.stack([base + (b & 1) + (b >> 1 & 1) * nphi + (b >> 2) * nphi * nt
                               for b in tet], -1)
            a = v[vid[:, 0]]
            e1, e2, e3, ep = v[vid[:, 1]] - a, v[vid[:, 2]] - a, v[vid[:, 3]] - a, p[at] - a
            c23 = torch.linalg.cross(e2, e3)
            det = (e1 * c23).sum(-1)
            b1 = (ep * c23).sum(-1) / det
            b2 = (e1 * torch.linalg.cross(ep, e3)).sum(-1) / det
            b3 = (e1 * torch.linalg.cross(e2, ep)).sum(-1) / det
            b0 = 1 - b1 - b2 - b3
            w = torch.stack([b0, b1, b2, b3], -1)
            hit = (w >= 0).all(-1) & (number + j < best[at])
            best[at[hit]] = number[hit] + j
            ids[at[hit]], wts[at[hit]] = vid[hit], w[hit]
    found = best < 1 << 62
    flat = x.reshape(x.shape[0], -1).to(torch.complex128 if x.is_complex() else torch.float64)
    if case["nearest"]:
        val = flat[:, ids.gather(1, wts.argmax(-1, keepdim=True))[:, 0]] * found
    else:
        val = torch.zeros((x.shape[0], nq), dtype=flat.dtype, device=_dev())
        for j in range(4):
            val += flat[:, ids[:, j]] * wts[:, j]
    return val.reshape((x.shape[0],) + tuple(q.shape[:-1]))


def exact(case, seed):
    if case["kind"] == "das":
        geo, x, target = _das_inputs(case, seed)
        wavenum = 2 * math.pi * F0 / FS if case["data"][0] == "c" else 0.0
        grad = {"forward": None, "step": lambda out: 2 * (out - target.double()),
                "autograd": lambda out: target}[case["mode"]]
        r = _das_exact(_natural(case, x), geo, wavenum=wavenum, scale=case["scale"], grad_out=grad)
        if grad is None:
            return r
        out, gx, go, gw, gs = r
        gx = gx.transpose(1, 2) if case["trailing"] else gx
        return [out, gx, go, gw] if case["mode"] == "autograd" else [out, gx, go, gs]
    if case["kind"] == "batched":
        return [_das_exact(q["x"], dict(q, srcdir=None, table=q["sparse_indices"]))
                for q in _batched_inputs(case, seed)]
    if case["kind"] == "rank":
        x = _rank_inputs(case, seed)
        x = x.to(torch.complex128 if x.is_complex() else torch.float64)
        gram = x @ x.mH
        u = torch.linalg.eigh(gram.cpu()).eigenvectors.flip(-1).to(_dev())
        p = min(x.shape)
        u = u[:, case["start"]:case["stop"] or p]
        return u @ (u.mH @ x)
    if case["kind"] == "interp":
        return _interp_exact(case, *_interp_inputs(case, seed))
    src, k, x, dst = (t.to(torch.complex128 if t.is_complex() else torch.float64)
                      for t in _greens_inputs(case, seed))
    flat = dst.reshape(-1, 3)
    out = torch.empty((case["events"], flat.shape[0], case["freqs"]), dtype=torch.complex128,
                      device=_dev())
    step = max(1, (1 << 26) // (case["sources"] * case["freqs"]))
    xf = x.permute(2, 1, 0).contiguous()                       # (freqs, sources, events)
    for a in range(0, flat.shape[0], step):
        r = torch.linalg.vector_norm(flat[a:a + step, None] - src[None], dim=-1)
        e = torch.polar((1 / r).expand(case["freqs"], *r.shape).contiguous(), k[:, None, None] * r)
        out[:, a:a + step] = torch.matmul(e, xf).permute(2, 1, 0)
    return out.reshape((case["events"],) + tuple(dst.shape[:-1]) + (case["freqs"],))
