"""The forward for few frames (das_few.hip) against the FP64 oracle and the plain kernels (GPU).

Tolerance: the kernel's delays are exact to 2^-31 of a sample and its sums are FP32, so FP32
storage keeps the forward's 1e-5 rel-L2 against the FP64 oracle; 16-bit storage is compared
with the oracle on the rounded data at the same bound.
"""
import numpy as np
import pytest

import oracle
from ffdas_amd import workloads as W
from tests.helpers import oracle_args, rel_l2, to_dev

pytestmark = pytest.mark.gpu


def _run(d, **kw):
    import ffdas_amd
    a = dict(d)
    si = a.pop("sparse_indices", None)
    geo = [a.pop(k) for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
    if si is not None:
        return ffdas_amd.das_sparse(*geo, si, **a, **kw)
    return ffdas_amd.das(*geo, **a, **kw)


# slots: below a group, a group, a round of 8 and its remainders, rounds of 16
@pytest.mark.parametrize("K", [1, 2, 3, 5, 8, 9, 16, 19, 33])
@pytest.mark.parametrize("B", [1, 2, 3])
@pytest.mark.parametrize("kind", ["f32", "f16", "c32", "sparse", "cone"])
def test_parity(dev, K, B, kind):
    import torch
    cplx, sparse = kind == "c32", kind == "sparse"
    w = W.small_random(seed=K + 40 * B, B=B, C=19, T=K, S=83, N=(5, 3, 7) if K % 2 else (13, 11),
                       K=K, complex_iq=cplx, srcdir=kind == "cone", sparse=sparse)
    if sparse:                                    # indices that select nothing
        w.sparse_indices.flat[::7] = -1
        w.sparse_indices.flat[1::11] = K
    scale = 1.0 if K % 3 else 1.03
    d = to_dev(w, dev, torch.float16 if kind == "f16" else None)
    args, kw = oracle_args(w)
    if kind == "f16":
        args = (w.x.astype(np.float16).astype(np.float64),) + args[1:]
    ref = oracle.das(*args, scale=scale, **kw)
    assert rel_l2(_run(d, scale=scale).cpu().numpy(), ref) < 1e-5


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("shape", [(1,), (64,), (65,), (3, 1, 129), (9, 4, 5)])
def test_strided_rows_and_grids(dev, cplx, shape):
    """Rows in (transmit, channel) order with gaps, odd sample counts, grids off the tiles."""
    import torch
    w = W.small_random(seed=3, B=1, C=7, T=4, S=61, N=shape, complex_iq=cplx)
    d = to_dev(w, dev)
    big = torch.zeros((1, 4, 9, 67), dtype=d["x"].dtype, device=dev)
    big[:, :, :7, :61] = d["x"].transpose(1, 2)
    d["x"] = big[:, :, :7, :61]
    args, kw = oracle_args(w)
    assert rel_l2(_run(d, channels_trailing=True).cpu().numpy(), oracle.das(*args, **kw)) < 1e-5


@pytest.mark.parametrize("where", ["offsets", "weights", "dstpos", "srcpos"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), 3e38, 1e30, -6e6,
                                   5e6, 1e-35])
def test_terms_beyond_fixed_point(dev, where, value):
    """Delays, weights and positions that the fixed-point tap does not hold give what the plain
    kernels give, not-a-numbers included."""
    import torch
    import ffdas_amd
    w = W.small_random(seed=9, B=2, C=6, T=5, S=96, N=(6, 23))
    d = to_dev(w, dev)
    t = d[where].clone()
    t.view(-1)[[3, 17 % t.numel()]] = value
    d[where] = t
    got = _run(d).cpu().numpy()
    ref = _run(d, algorithm=ffdas_amd.Algorithm.ALG1).cpu().numpy()
    fine = np.isfinite(ref)
    if where == "weights" and value == 3e38:
        # whether the sum of terms near the largest float overflows depends on their order,
        # which the two kernels do not share: the two voxels with that weight say nothing
        fine = np.ones(ref.shape, bool)
        fine.reshape(2, -1)[:, [3, 17]] = False
        assert np.isfinite(got[fine]).all() and np.isfinite(ref[fine]).all()
    else:
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got[~fine & ~np.isnan(ref)], ref[~fine & ~np.isnan(ref)])
    if fine.any():
        # a weight near the largest float dwarfs the rest: compare voxel by voxel
        got, ref = got[fine].astype(np.float64), ref[fine].astype(np.float64)
        scale = np.maximum(np.abs(ref), np.median(np.abs(ref)))
        assert np.max(np.abs(got - ref) / scale) < 1e-4
    assert torch.isfinite(_run(to_dev(w, dev))).all()


def test_chunked_tile_order_covers_every_voxel(dev):
    """Grids of a few thousand tiles, whose blocks are dealt to the XCDs in chunks."""
    w = W.small_random(seed=5, B=1, C=2, T=1, S=64, N=(67, 66, 41))
    args, kw = oracle_args(w)
    assert rel_l2(_run(to_dev(w, dev)).cpu().numpy(), oracle.das(*args, **kw)) < 1e-5
