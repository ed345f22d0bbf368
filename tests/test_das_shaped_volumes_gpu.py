"""Volumes with taps enough for shaped tiles, and just too few for them (GPU): forward and parameter
adjoint against the FP64 oracle, with the depth, and so the thin side of the tiles, along each axis.

Tolerance: 1e-5 rel-L2 for the image and the weights' gradient, as in the other tests of these kernels.
The delays' gradient jumps where a tap falls on a whole sample, and of the half million taps here some
fall within 5e-8 of one; it comes from the same taps and is compared where there are fewer."""
import numpy as np
import pytest

import oracle
from ffdas_amd import workloads as W
from tests.helpers import oracle_args, rel_l2, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(9, 17, 10), (5, 6, 33)])
@pytest.mark.parametrize("C,K", [(127, 4), (128, 4), (103, 5)])
@pytest.mark.parametrize("B,cplx", [(4, False), (8, False), (16, False), (4, True)])
def test_frames(dev, grid, C, K, B, cplx):
    import torch
    import ffdas_amd
    for axis in range(3):
        w = W.small_random(seed=axis, B=B, C=C, T=K, S=64, N=grid, complex_iq=cplx)
        z = np.sort(w.dstpos[..., 2], axis=axis)
        w.dstpos[..., 2] = z
        w.offsets[:] = 0.5 * z + w.offsets * 0.01
        d = to_dev(w, dev)
        geo = [d[k] for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
        args, kw = oracle_args(w)
        got = ffdas_amd.das(*geo, wavenum=w.wavenum).cpu().numpy()
        assert rel_l2(got, oracle.das(*args, **kw)) < 1e-5
        g = np.random.default_rng(1).standard_normal((B,) + grid).astype(np.float32)
        if cplx:
            g = (g + 1j * g[::-1]).astype(np.complex64)
        _, _, gw, _ = ffdas_amd.das_backward(*geo, torch.from_numpy(g).to(dev), wavenum=w.wavenum, need_x=False)
        ref = oracle.das_adjoint(*args, g, **kw)
        assert rel_l2(gw.cpu().numpy(), ref["grad_weights"]) < 1e-5


@pytest.mark.parametrize("K", [7, 8])
@pytest.mark.parametrize("B,cplx", [(1, False), (2, False), (1, True)])
def test_few_frames(dev, K, B, cplx):
    import ffdas_amd
    for axis in range(3):
        w = W.small_random(seed=axis, B=B, C=1024, T=K, S=64, N=(5, 9, 10), complex_iq=cplx)
        z = np.sort(w.dstpos[..., 2], axis=axis)
        w.dstpos[..., 2] = z
        w.offsets[:] = 0.5 * z + w.offsets * 0.01
        d = to_dev(w, dev)
        got = ffdas_amd.das(*[d[k] for k in ("x", "srcpos", "dstpos", "offsets", "weights")], wavenum=w.wavenum)
        args, kw = oracle_args(w)
        assert rel_l2(got.cpu().numpy(), oracle.das(*args, **kw)) < 1e-5
