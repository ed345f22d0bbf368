"""greens at the edges of its MFMA tiles (16 targets, 8 events, 8 frequencies, 8 staged sources)
against the FP64 oracle (GPU).

Tolerance: 2e-5 of the sum's scale, as the other greens tests: the phase k r and the distance
are FP32, a few 1e-7 relative each, at phases up to some tens of radians here."""
import numpy as np
import pytest

import oracle.greens as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("events", [2, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("sources", [1, 3, 8, 9, 20])
@pytest.mark.parametrize("freqs,targets", [(1, 63), (7, 16), (8, 1), (9, 65), (16, 17)])
def test_tile_edges(dev, events, sources, freqs, targets):
    import torch
    import ffdas_amd
    rng = np.random.default_rng(events * 1000 + sources * 10 + freqs)
    src = rng.standard_normal((sources, 3)).astype(np.float32)
    dst = rng.standard_normal((targets, 3)).astype(np.float32)
    k = rng.uniform(1.0, 10.0, freqs).astype(np.float32)
    x = (rng.standard_normal((events, sources, freqs))
         + 1j * rng.standard_normal((events, sources, freqs))).astype(np.complex64)
    t = lambda a: torch.from_numpy(a).to(dev)
    ref = G.greens(src, k, x, dst)
    for xx in (t(x), t(x).to(torch.complex32)):
        want = ref if xx.dtype == torch.complex64 else G.greens(
            src, k, xx.to(torch.complex64).cpu().numpy(), dst)
        got = ffdas_amd.greens(t(src), t(k), xx, t(dst)).cpu().numpy()
        r = np.linalg.norm(dst[:, None] - src[None], axis=-1)
        scale = np.einsum("bsf,ts->btf", np.abs(x), 1.0 / r)      # the terms' magnitudes
        assert np.max(np.abs(got - want) / scale) < 2e-5


def test_coincident_and_non_finite(dev):
    """A target on a source and a non-finite field value give what their own sums give, and
    leave the other events, targets and frequencies alone."""
    import torch
    import ffdas_amd
    rng = np.random.default_rng(1)
    src = rng.standard_normal((5, 3)).astype(np.float32)
    dst = rng.standard_normal((20, 3)).astype(np.float32)
    dst[7] = src[2]
    x = (rng.standard_normal((3, 5, 9)) + 1j * rng.standard_normal((3, 5, 9))).astype(np.complex64)
    x[1, 4, 3] = np.inf
    k = rng.uniform(1.0, 10.0, 9).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    got = ffdas_amd.greens(t(src), t(k), t(x), t(dst)).cpu().numpy()
    bad = ~(np.isfinite(got.real) & np.isfinite(got.imag))
    want = np.zeros_like(bad)
    want[:, 7] = True
    want[1, :, 3] = True
    assert np.array_equal(bad, want)
