"""Location by cells against the point-by-point scan, and the frame chunks of the evaluation
against single frames (GPU).  Both comparisons are bit for bit: the candidates, the FP32 test and
the order of the weighted sum are the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grid(rng, nz, ny, nx, jitter):
    z, y, x = np.meshgrid(np.linspace(0.2, 1, nz), np.linspace(-.6, .6, ny),
                          np.linspace(-.6, .6, nx), indexing="ij")
    g = np.stack([z * np.sin(x) * np.cos(y), z * np.sin(y), z * np.cos(x) * np.cos(y)], -1)
    return (g + jitter * rng.standard_normal(g.shape) / max(nz, ny, nx)).astype(np.float32)


def _points(rng, g, n):
    flat = g.reshape(-1, 3)
    lo, hi = flat.min(0), flat.max(0)
    q = rng.uniform(lo - 0.02, hi + 0.02, (n, 3)).astype(np.float32)
    k = n // 5
    q[:k] = flat[rng.integers(0, len(flat), k)]                            # on vertices
    q[k:2 * k] = 0.5 * (flat[rng.integers(0, len(flat) - 1, k)] + flat[1:][rng.integers(0, len(flat) - 1, k)])
    q[2 * k:2 * k + 3] = [[np.nan, 0, 0], [np.inf, 0, 0], [-np.inf, 0, 0]]
    return q


# fine grids with few points to coarse grids with many: every split of runs and points over lanes
@pytest.mark.parametrize("shape,n", [((2, 2, 2), 70000), ((3, 4, 5), 200001), ((9, 5, 7), 1000000),
                                     ((40, 17, 23), 300000), ((60, 50, 40), 5000), ((30, 2, 31), 777),
                                     ((1, 9, 9), 500), ((4, 6, 1), 500)])
@pytest.mark.parametrize("mode", ["linear", "nearest"])
def test_cells_match_point_scan(dev, monkeypatch, shape, n, mode):
    import torch
    import ffdas_amd
    rng = np.random.default_rng(sum(shape) + n)
    g = _grid(rng, *shape, jitter=0.3 if n % 2 else 0.0)
    t = lambda a: torch.from_numpy(a).to(dev)
    q, x = t(_points(rng, g, n)), t(rng.standard_normal(shape).astype(np.float32))
    cells = ffdas_amd.interpolate(t(g), x, q, mode=mode, fill=7.5)
    monkeypatch.setenv("FFDAS_INTERP_LOCATE", "point")
    scan = ffdas_amd.interpolate(t(g), x, q, mode=mode, fill=7.5)
    assert torch.equal(cells, scan)
    if min(shape) > 1:
        assert (cells != 7.5).float().mean() > 0.2


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 4097, 50000])
def test_queue_fills_and_drains(dev, monkeypatch, n):
    """Two cells in turn: the lanes of a wave queue none, some or all of their points a step, across
    the queue's own length."""
    import torch
    import ffdas_amd
    rng = np.random.default_rng(n)
    z, y, x = np.meshgrid([0., 1.], [0., 1.], [0., 1., 2.], indexing="ij")
    g = np.stack([x, y, z + 0.3 * x], -1).astype(np.float32)       # sheared: half the box is empty
    q = rng.uniform([0, 0, 0], [2, 1, 1.6], (n, 3)).astype(np.float32)
    q[::3, 0] = rng.uniform(0.4, 0.6, len(q[::3]))
    t = lambda a: torch.from_numpy(a).to(dev)
    v = t(rng.standard_normal(g.shape[:3]).astype(np.float32))
    cells = ffdas_amd.interpolate(t(g), v, t(q), fill=7.5)
    monkeypatch.setenv("FFDAS_INTERP_LOCATE", "point")
    assert torch.equal(cells, ffdas_amd.interpolate(t(g), v, t(q), fill=7.5))


@pytest.mark.parametrize("dtype", ["float32", "complex64", "float64", "complex128"])
@pytest.mark.parametrize("frames", [1, 2, 3, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("n", [64, 5001])          # rows of whole cache lines, and not
@pytest.mark.parametrize("mode", ["linear", "nearest"])
def test_frame_chunks_match_single_frames(dev, dtype, frames, n, mode):
    import torch
    import ffdas_amd
    rng = np.random.default_rng(frames)
    g = _grid(rng, 9, 7, 8, 0.2)
    x = rng.standard_normal((frames, 9, 7, 8, 2))
    x = (x[..., 0] + 1j * x[..., 1] if "complex" in dtype else x[..., 0]).astype(dtype)
    t = lambda a: torch.from_numpy(a).to(dev)
    plan, q, xt = ffdas_amd.Interpolator(t(g), mode=mode), t(_points(rng, g, n)), t(x)
    plan.preprocess(q)
    out = plan(xt, q, fill=-3.0)
    ref = torch.stack([plan(xt[b], q, fill=-3.0) for b in range(frames)])
    assert torch.equal(out, ref)
    # an output off the 16-byte and cache-line boundaries
    buf = torch.full((frames * n + 1,), 5.0, dtype=xt.dtype, device=dev)
    view = buf[1:].view(frames, n)
    plan(xt, q, fill=-3.0, out=view)
    assert torch.equal(view, ref) and buf[0] == 5.0


@pytest.mark.parametrize("frames", [1, 2, 16])
@pytest.mark.parametrize("mode", ["linear", "nearest"])
@pytest.mark.parametrize("kept", [True, False])
@pytest.mark.parametrize("shift", [0, 100])
def test_output_over_the_input(dev, frames, mode, kept, shift):
    """A volume warped in place, wholly or partly: every value is read before it is overwritten."""
    import torch
    import ffdas_amd
    rng = np.random.default_rng(frames + shift)
    nz, ny, nx = 40, 41, 42
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    g = np.stack([x, y, z], -1).astype(np.float32)
    q = g[::-1, ::-1, ::-1].copy()                      # each point reads the far end of the volume
    t = lambda a: torch.from_numpy(a).to(dev)
    v = t(rng.standard_normal((frames, nz, ny, nx)).astype(np.float32))
    plan, q = ffdas_amd.Interpolator(t(g), mode=mode), t(q)
    if kept:
        plan.preprocess(q)
    ref = plan(v, q)
    buf = torch.zeros(v.numel() + shift, dtype=v.dtype, device=dev)
    xin, out = buf[:v.numel()].view(v.shape), buf[shift:].view(v.shape)
    xin.copy_(v)
    plan(xin, q, out=out)
    assert torch.equal(out, ref)
