"""greens with two events where the VALU kernel's workgroups fill the rounds they take, and where they
just do not (GPU). 668 workgroups of 256 targets and 16 frequencies are 0.87 of a round.

Tolerance: 2e-5 of the terms' magnitudes against the FP64 oracle, as the other greens tests."""
import numpy as np
import pytest

import oracle.greens as G
from tests.test_greens_few_freqs_gpu import _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sources", [63, 64])
@pytest.mark.parametrize("freqs,targets", [(64, 42753), (64, 42752), (61, 42753), (65, 34000)])
def test_parity(dev, sources, freqs, targets):
    import torch
    import ffdas_amd
    (src, k, x, dst), t = _problem(dev, 2, sources, freqs, targets)
    some = np.r_[0:300, targets - 300:targets]          # the oracle's targets: the first and the last tiles
    scale = np.abs(x).transpose(0, 2, 1) @ (1.0 / np.linalg.norm(dst[some, None] - src[None], axis=-1)).T
    for xx in (t[2], t[2].to(torch.complex32)):
        want = G.greens(src, k, xx.to(torch.complex64).cpu().numpy(), dst[some])
        got = ffdas_amd.greens(t[0], t[1], xx, t[3]).cpu().numpy()[:, some]
        assert np.max(np.abs(got - want) / scale.transpose(0, 2, 1)) < 2e-5
