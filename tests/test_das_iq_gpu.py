"""The complex forward with a rotation per slot and one per channel, against the FP64 oracle and the
plain kernels (GPU).

Tolerance: each rotation is good to 1e-7 and their product and the FP32 sums stay well inside the
1e-5 rel-L2 that the complex forward has against the FP64 oracle; half2 data is compared with the
oracle on the rounded data at the same bound.
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


@pytest.mark.parametrize("B", [1, 3, 4, 8, 16, 21])
@pytest.mark.parametrize("K", [1, 2, 7, 8, 9, 17])
@pytest.mark.parametrize("kind", ["c32", "c16", "sparse", "cone"])
def test_parity(dev, B, K, kind):
    import torch
    sparse = kind == "sparse"
    w = W.small_random(seed=B + 30 * K, B=B, C=11, T=K, S=83, N=(5, 3, 7) if K % 2 else (13, 11),
                       K=K, complex_iq=True, srcdir=kind == "cone", sparse=sparse)
    if sparse:                                    # indices that select nothing
        w.sparse_indices.flat[::7] = -1
        w.sparse_indices.flat[1::11] = K
    scale = 1.0 if K % 3 else 0.97
    d = to_dev(w, dev)
    args, kw = oracle_args(w)
    if kind == "c16":
        xr = torch.view_as_real(d["x"]).to(torch.float16)
        d["x"] = torch.view_as_complex(xr)
        args = (torch.view_as_complex(xr.to(torch.float64).cpu()).numpy(),) + args[1:]
    ref = oracle.das(*args, scale=scale, **kw)
    assert rel_l2(_run(d, scale=scale).cpu().numpy(), ref) < 1e-5


@pytest.mark.parametrize("B", [2, 4, 8])
@pytest.mark.parametrize("where", ["offsets", "weights", "dstpos", "srcpos"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), -6e6, 5e6])
def test_terms_beyond_fixed_point(dev, B, where, value):
    """Delays, weights and positions that the fixed-point tap does not hold give what the plain
    kernels give, not-a-numbers included."""
    import ffdas_amd
    w = W.small_random(seed=9, B=B, C=6, T=5, S=96, N=(6, 23), complex_iq=True)
    d = to_dev(w, dev)
    t = d[where].clone()
    t.view(-1)[[3, 17 % t.numel()]] = value
    d[where] = t
    got = _run(d).cpu().numpy()
    ref = _run(d, algorithm=ffdas_amd.Algorithm.ALG1).cpu().numpy()
    fine = np.isfinite(ref)
    assert np.array_equal(np.isfinite(got), fine)
    if fine.any():                                # one bad channel spoils every voxel
        got, ref = got[fine], ref[fine]
        scale = np.maximum(np.abs(ref), np.median(np.abs(ref)))
        assert np.max(np.abs(got - ref) / scale) < 1e-4


@pytest.mark.parametrize("B", [1, 2, 8])
@pytest.mark.parametrize("cplx", [False, True])
def test_slot_that_selects_nothing_has_no_weight(dev, B, cplx):
    """The weight of a slot whose index selects no transmit is not read, whatever it holds."""
    w = W.small_random(seed=4, B=B, C=6, T=5, S=96, N=(6, 23), K=3, sparse=True, complex_iq=cplx)
    w.sparse_indices.flat[::5] = -1
    args, kw = oracle_args(w)
    ref = oracle.das(*args, **kw)
    for value in (np.nan, np.inf, -np.inf):
        w.weights.flat[::5] = value
        assert rel_l2(_run(to_dev(w, dev)).cpu().numpy(), ref) < 1e-5
