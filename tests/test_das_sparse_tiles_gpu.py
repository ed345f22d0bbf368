"""Sparse compounding of volumes large enough that the kernels shape their tiles, give a workgroup several
and deal them to the XCDs in chunks, against the FP64 oracle (GPU).  The tile counts are no multiples of a
workgroup's tiles nor of a round of chunks, and each axis in turn is the steep one.
Tolerance: 1e-5 rel-L2, as every FP32 forward."""
import numpy as np
import pytest

import oracle
from ffdas_amd import workloads as W
from tests.helpers import oracle_args, rel_l2, to_dev

pytestmark = pytest.mark.gpu

GRIDS = [(33, 30, 29), (64, 20, 17), (25, 31, 27)]      # 576, 400 and 392 cubes


def _problem(seed, grid, axis, B, C, cplx=False):
    w = W.small_random(seed=seed, B=B, C=C, T=5, S=96, N=grid, K=3, sparse=True, complex_iq=cplx)
    z = np.sort(w.dstpos[..., 2], axis=axis)
    w.dstpos[..., 2] = z
    w.offsets[:] = 0.4 * z + 0.02 * w.offsets
    w.sparse_indices.flat[::17] = -1
    return w


def _check(w, out):
    args, kw = oracle_args(w)
    assert rel_l2(out.cpu().numpy(), oracle.das(*args, **kw)) < 1e-5


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("B,C,cplx", [(4, 2, False), (8, 3, False), (5, 1, False), (4, 3, True), (2, 3, False)])
def test_one_problem(dev, grid, axis, B, C, cplx):
    import ffdas_amd
    w = _problem(axis, grid, axis, B, C, cplx)
    d = to_dev(w, dev)
    si = d.pop("sparse_indices")
    geo = [d.pop(k) for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
    _check(w, ffdas_amd.das_sparse(*geo, si, **d))


@pytest.mark.parametrize("C", [1, 2, 3])
def test_batched(dev, C):
    """The three grids with each steep axis, and small ones between them, in one launch."""
    import ffdas_amd
    ws = [_problem(3 * i + a, g, a, 4 + i, C) for i, g in enumerate(GRIDS) for a in range(3)]
    ws[2:2] = [_problem(20, (9, 5, 7), 0, 4, C), _problem(21, (70, 90, 2), 1, 6, C)]
    outs = ffdas_amd.das_batched([to_dev(w, dev) for w in ws])
    for w, o in zip(ws, outs):
        _check(w, o)
