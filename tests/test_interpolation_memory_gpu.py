"""What interpolate keeps of the GPU's memory between calls (GPU): the handle's workspace, bounded, and a
plan's own lookup; the scratch of a large point set goes back with the call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the kept scratch (256 MiB and a quarter of headroom), and what the allocators round up to
KEPT = 400 << 20


def _setup(dev, n):
    import torch
    z, y, x = torch.meshgrid(*[torch.linspace(0, 1, 24, device=dev)] * 3, indexing="ij")
    grid = torch.stack([x, y, z], -1).contiguous()
    g = torch.Generator(device=dev).manual_seed(1)
    q = torch.rand(n, 3, device=dev, generator=g)
    v = torch.rand(24, 24, 24, device=dev, generator=g)
    return grid, v, q, torch.empty(n, device=dev)


@pytest.mark.parametrize("preprocess", [False, True])
def test_large_point_set_leaves_little(dev, preprocess):
    import torch
    import ffdas_amd
    n = 24 << 20                      # scratch and lookup take 38 bytes a point, 960 MB
    grid, v, q, out = _setup(dev, n)
    with torch.cuda.stream(torch.cuda.Stream()):     # a handle of its own
        small = _setup(dev, 1000)
        ffdas_amd.interpolate(small[0], small[1], small[2], out=small[3])
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        before = torch.cuda.mem_get_info()[0]
        plan = ffdas_amd.Interpolator(grid)
        for _ in range(2):
            if preprocess:
                plan.preprocess(q)
            plan(v, q, out=out)
        plan.close()
        torch.cuda.synchronize()
        assert before - torch.cuda.mem_get_info()[0] < KEPT
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("n", [1000, 6_000_000, 9_000_000])
@pytest.mark.parametrize("frames", [1, 3])
def test_sizes_about_the_kept_scratch(dev, monkeypatch, n, frames):
    """Calls on either side of the bound, in both orders, give the same values."""
    import torch
    import ffdas_amd
    grid, v, q, _ = _setup(dev, n)
    v = v.expand(frames, 24, 24, 24).contiguous() + torch.arange(frames, device=dev).reshape(-1, 1, 1, 1)
    with torch.cuda.stream(torch.cuda.Stream()):
        first = ffdas_amd.interpolate(grid, v, q)
        ffdas_amd.interpolate(grid, v, q[:100])
        plan = ffdas_amd.Interpolator(grid)
        plan.preprocess(q)
        kept = plan(v, q)
        torch.cuda.synchronize()
        monkeypatch.setenv("FFDAS_INTERP_LOCATE", "point")
        scan = ffdas_amd.interpolate(grid, v, q)
        torch.cuda.synchronize()
    assert torch.equal(first, scan) and torch.equal(kept, scan)
