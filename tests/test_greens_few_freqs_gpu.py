"""greens with two to four events, few frequencies and many targets, whose sums stay on the VALU (GPU).

Tolerance: 2e-5 of the sum's scale against the FP64 oracle, as the other greens tests.  Time: the second to
fourth event share the sines and cosines of the first and add two multiply-adds each, so four times
one event's time is far above theirs (1.7 and 2.1 times; 7.8 times on the MFMA, which forms eight
frequencies and eight events whatever there are)."""
import numpy as np
import pytest

import oracle.greens as G

pytestmark = pytest.mark.gpu


def _problem(dev, events, sources, freqs, targets):
    import torch
    rng = np.random.default_rng(events * 100 + sources * 10 + freqs)
    src = rng.standard_normal((sources, 3)).astype(np.float32)
    dst = (rng.standard_normal((targets, 3)) + 4).astype(np.float32)
    k = rng.uniform(1.0, 10.0, freqs).astype(np.float32)
    x = (rng.standard_normal((events, sources, freqs))
         + 1j * rng.standard_normal((events, sources, freqs))).astype(np.complex64)
    return (src, k, x, dst), [torch.from_numpy(a).to(dev) for a in (src, k, x, dst)]


@pytest.mark.parametrize("events", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("freqs", [1, 3, 5, 7, 9])
@pytest.mark.parametrize("targets", [65536 + 1, 262144 - 3])
def test_parity(dev, events, freqs, targets):
    import torch
    import ffdas_amd
    (src, k, x, dst), t = _problem(dev, events, 3, freqs, targets)
    r = np.linalg.norm(dst[:, None] - src[None], axis=-1)
    scale = np.abs(x).transpose(0, 2, 1) @ (1.0 / r).T            # the terms' magnitudes
    for xx in (t[2], t[2].to(torch.complex32)):
        want = G.greens(src, k, xx.to(torch.complex64).cpu().numpy(), dst)
        got = ffdas_amd.greens(t[0], t[1], xx, t[3]).cpu().numpy()
        assert np.max(np.abs(got - want) / scale.transpose(0, 2, 1)) < 2e-5


@pytest.mark.parametrize("events", [2, 4])
def test_single_frequency_time(dev, events):
    import torch
    import ffdas_amd

    def ms(n):
        _, t = _problem(dev, n, 128, 1, 1 << 20)
        best = []
        for _ in range(8):
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            for _ in range(5):
                ffdas_amd.greens(*t)
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        return min(best)

    assert ms(events) < 4 * ms(1)
