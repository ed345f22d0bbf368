"""Volumes in tiles thin along the steepest axis, and several tiles a workgroup, against the FP64
oracle (GPU).  Tolerance: 1e-5 rel-L2, as every FP32 forward and adjoint."""
import numpy as np
import pytest

import oracle
from ffdas_amd import workloads as W
from tests.helpers import oracle_args, rel_l2, to_dev

pytestmark = pytest.mark.gpu

GRIDS = [(2, 2, 2), (9, 5, 7), (3, 17, 2), (2, 3, 33), (33, 3, 2), (16, 9, 8), (2, 3, 4, 5)]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("B,C", [(1, 3), (4, 9), (16, 16)])
def test_volume_tiles(dev, grid, sparse, B, C):
    """The random positions of each seed put the steepest axis first, in the middle or last."""
    import ffdas_amd
    for seed in range(4):
        w = W.small_random(seed=seed, B=B, C=C, T=5, S=64, N=grid, K=3 if sparse else None,
                           sparse=sparse)
        d = to_dev(w, dev)
        si = d.pop("sparse_indices", None)
        geo = [d.pop(k) for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
        out = ffdas_amd.das_sparse(*geo, si, **d) if sparse else ffdas_amd.das(*geo, **d)
        args, kw = oracle_args(w)
        assert rel_l2(out.cpu().numpy(), oracle.das(*args, **kw)) < 1e-5, seed
    g = np.random.default_rng(1).standard_normal(out.shape).astype(np.float32)
    import torch
    gx, go, gw, gs = ffdas_amd.das_backward(*geo, torch.from_numpy(g).to(dev), sparse_indices=si)
    ref = oracle.das_adjoint(*args, g, sparse_indices=w.sparse_indices)
    assert rel_l2(gx.cpu().numpy(), ref["grad_x"]) < 1e-5
    assert rel_l2(go.cpu().numpy(), ref["grad_offsets"]) < 1e-4
    assert rel_l2(gw.cpu().numpy(), ref["grad_weights"]) < 1e-5


def test_batched_mixes_tile_counts(dev):
    """Problems whose tiles do not fill whole workgroups, dense and sparse, in one call."""
    import ffdas_amd
    ws = [W.small_random(seed=i, B=8, C=6 + i, T=4, S=64, N=g, K=3 if i % 2 else None,
                         sparse=bool(i % 2)) for i, g in enumerate(GRIDS + [(13, 9), (70,)])]
    outs = ffdas_amd.das_batched([to_dev(w, dev) for w in ws])
    for w, o in zip(ws, outs):
        args, kw = oracle_args(w)
        assert rel_l2(o.cpu().numpy(), oracle.das(*args, **kw)) < 1e-5


def test_orientations_cover_the_grid():
    """Every voxel is in one tile of every shape and orientation (the kernels' index arithmetic,
    on the CPU)."""
    for A, H, Wd in [(2, 2, 2), (9, 5, 7), (3, 17, 2), (5, 16, 33)]:
        for steep in range(3):
            for t in [(1, 8, 8), (1, 4, 16), (1, 16, 4), (2, 8, 4), (2, 4, 8), (4, 4, 4)]:
                ta, th, tw = {0: t, 1: (t[1], t[0], t[2]), 2: (t[1], t[2], t[0])}[steep]
                nta, nth, ntw = -(-A // ta), -(-H // th), -(-Wd // tw)
                seen = np.zeros(A * H * Wd, int)
                for tile in range(nta * nth * ntw):
                    if steep == 2:
                        ih, rest = tile % nth, tile // nth
                        ia, iw = rest % nta, rest // nta
                    else:
                        iw, rest = tile % ntw, tile // ntw
                        nin = nta if steep == 1 else nth
                        ia, ih = (rest % nin, rest // nin) if steep == 1 else (rest // nin, rest % nin)
                    lane = np.arange(64)
                    w = iw * tw + lane % tw
                    h = ih * th + lane // tw % th
                    a = ia * ta + lane // (tw * th)
                    ok = (w < Wd) & (h < H) & (a < A)
                    np.add.at(seen, ((a * H + h) * Wd + w)[ok], 1)
                assert (seen == 1).all()
