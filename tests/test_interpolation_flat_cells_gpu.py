"""Location by cells where cells are so flat that the FP32 weights of their tetrahedra mean little (GPU): a
point well outside a cell may pass its test, and the scan over the bin's tetrahedra takes it.  Bit for
bit the point-by-point scan's values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _slab(rng, shape, thickness, offset):
    """A grid whose layers lie `thickness` apart, turned out of the axes."""
    z, y, x = np.meshgrid(*[np.linspace(0, 1, n) for n in shape], indexing="ij")
    turn = np.linalg.qr(rng.standard_normal((3, 3)))[0]
    place = lambda p: (offset + p * [1, 1, thickness * shape[0]]) @ turn.T
    g = place(np.stack([x, y, z], -1))
    q = rng.uniform(-0.05, 1.05, (200000, 3))
    q[::2, 2] = rng.choice([0.0, 0.25, 0.5, 1.0], len(q[::2]))
    return g.astype(np.float32), place(q).astype(np.float32)


@pytest.mark.parametrize("thickness", [0.0, 1e-7, 1e-6, 1e-5, 1e-4, 1e-2])
@pytest.mark.parametrize("shape", [(2, 150, 150), (5, 60, 60), (4, 200, 30)])
@pytest.mark.parametrize("mode", ["linear", "nearest"])
def test_matches_point_scan(dev, monkeypatch, shape, thickness, mode):
    import torch
    import ffdas_amd
    t = lambda a: torch.from_numpy(a).to(dev)
    for seed, offset in enumerate([0.0, 3.0, 20.0]):
        rng = np.random.default_rng(seed)
        g, q = _slab(rng, shape, thickness, offset)
        x = t(rng.standard_normal(shape).astype(np.float32))
        monkeypatch.delenv("FFDAS_INTERP_LOCATE", raising=False)
        cells = ffdas_amd.interpolate(t(g), x, t(q), mode=mode, fill=7.5)
        monkeypatch.setenv("FFDAS_INTERP_LOCATE", "point")
        scan = ffdas_amd.interpolate(t(g), x, t(q), mode=mode, fill=7.5)
        assert torch.equal(cells, scan), (seed, int((cells != scan).sum()))
