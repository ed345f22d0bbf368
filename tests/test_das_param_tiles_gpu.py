"""The parameter adjoint on volumes whose launch holds more workgroups than tiles (GPU): the gradients
against the FP64 oracle, the scale's above all, which sums over all workgroups, those without a tile included.

Tolerance: 1e-4 for the gradients of the delays and the scale, 1e-5 for the weights', as in the other
adjoint tests."""
import numpy as np
import pytest

import oracle
from ffdas_amd import workloads as W
from tests.helpers import oracle_args, rel_l2, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(2, 9, 17), (9, 2, 17), (17, 9, 2), (3, 17, 9), (17, 3, 9), (9, 17, 3)])
@pytest.mark.parametrize("B,C,cplx", [(4, 2, False), (8, 11, False), (16, 3, False), (4, 9, True)])
def test_gradients(dev, grid, B, C, cplx):
    import torch
    import ffdas_amd
    for axis in range(3):
        w = W.small_random(seed=axis, B=B, C=C, T=3, S=96, N=grid, complex_iq=cplx)
        # the depth, and so the steepest delays, along this axis
        z = np.sort(w.dstpos[..., 2], axis=axis)
        w.dstpos[..., 2] = z
        w.offsets[:] = 0.5 * z + w.offsets * 0.01
        d = to_dev(w, dev)
        geo = [d[k] for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
        g = np.random.default_rng(1).standard_normal((B,) + grid).astype(w.x.real.dtype)
        if cplx:
            g = (g + 1j * g[::-1]).astype(np.complex64)
        _, go, gw, gs = ffdas_amd.das_backward(*geo, torch.from_numpy(g).to(dev), wavenum=w.wavenum,
                                               scale=1.01, need_x=False)
        args, kw = oracle_args(w)
        ref = oracle.das_adjoint(*args, g, scale=1.01, **kw)
        assert rel_l2(go.cpu().numpy(), ref["grad_offsets"]) < 1e-4
        assert rel_l2(gw.cpu().numpy(), ref["grad_weights"]) < 1e-5
        assert abs(float(gs) - ref["grad_scale"]) < 1e-4 * max(1.0, abs(ref["grad_scale"]))

