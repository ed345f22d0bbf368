"""Location by cells where cells and points are far from even (GPU): coarse grids, rasters of a small part
of a grid, grids with cells much larger than the rest, more leftover work than its list holds.  Bit
for bit the point-by-point scan's values.

Time: an even raster is located at several hundred points a microsecond; 200 and half a millisecond for
the launches are asked of these (with the lanes of an average cell they take 5 to 30 times that)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(n, crowd=1.0):
    """n^3 vertices over the unit cube, all but the last plane along each axis within `crowd` of it."""
    a = np.linspace(0, 1, n)
    a[:-1] *= crowd
    z, y, x = np.meshgrid(a, a, a, indexing="ij")
    return np.stack([x, y, z], -1).astype(np.float32)


def _raster(n, lo, hi):
    a = np.linspace(lo, hi, n)
    z, y, x = np.meshgrid(a, a, a, indexing="ij")
    return np.stack([x, y, z], -1).astype(np.float32)


CASES = {
    "coarse": (_box(2), _raster(90, 0, 1)),
    "coarse, few points": (_box(3), _raster(15, 0, 1)),
    "zoomed": (_box(16), _raster(80, 0.5, 0.56)),
    "zoomed, fine": (_box(60), _raster(80, 0.31, 0.38)),
    "one bin": (_box(9), _raster(50, 0.5001, 0.5002)),
    "large cell": (_box(30, 0.2), _raster(70, 0, 1)),
    "large cell, zoomed": (_box(30, 0.2), _raster(60, 0.5, 0.6)),
    "more than the list": (_box(40, 0.01), _raster(27, 0.0, 0.009)),
    "corner": (_box(40, 0.01), _raster(60, 0.0, 0.02)),
}


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("mode", ["linear", "nearest"])
def test_matches_point_scan(dev, monkeypatch, case, mode):
    import torch
    import ffdas_amd
    g, q = CASES[case]
    rng = np.random.default_rng(len(case))
    h = np.diff(np.unique(g)).min()
    g = (g + 0.2 * h * rng.standard_normal(g.shape)).astype(np.float32)       # oblique cells
    t = lambda a: torch.from_numpy(a).to(dev)
    g, x, q = t(g), t(rng.standard_normal(g.shape[:3]).astype(np.float32)), t(q)
    print(case, mode, flush=True)
    cells = ffdas_amd.interpolate(g, x, q, mode=mode, fill=7.5)
    monkeypatch.setenv("FFDAS_INTERP_LOCATE", "point")
    scan = ffdas_amd.interpolate(g, x, q, mode=mode, fill=7.5)
    assert torch.equal(cells, scan)
    assert (cells != 7.5).float().mean() > 0.2


@pytest.mark.parametrize("case", ["coarse", "zoomed", "large cell", "large cell, zoomed"])
def test_time(dev, case):
    import torch
    import ffdas_amd
    g, q = (torch.from_numpy(a).to(dev) for a in CASES[case])
    plan = ffdas_amd.Interpolator(g)

    def ms():
        best = []
        for _ in range(4):
            torch.cuda.synchronize()
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            plan.preprocess(q)
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        return min(best)

    assert ms() < 0.5 + q[..., 0].numel() / 200e3
