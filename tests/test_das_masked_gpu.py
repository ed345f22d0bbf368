"""Voxels masked by an offset beyond every sample (GPU): the same image as the plain kernels form, for
about the price of the image without the mask.

Tolerance: 1e-5 rel-L2 against the plain kernels, as every FP32 forward has against the FP64 oracle.
Time: masked slots only do less; a quarter above the unmasked image is the scatter allowed for (a wave
that takes its taps one by one for them needs 1.45 to 2.7 times as long)."""
import pytest

from ffdas_amd import workloads as W
from tests.helpers import rel_l2, to_dev

pytestmark = pytest.mark.gpu


def _run(d, **kw):
    import ffdas_amd
    geo = [d[k] for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
    kw["wavenum"] = d.get("wavenum", 0.0)
    if "sparse_indices" in d:
        return ffdas_amd.das_sparse(*geo, d["sparse_indices"], **kw)
    return ffdas_amd.das(*geo, **kw)


def _ms(d):
    """The least of several runs of the forward kernels, by events."""
    import torch
    times = []
    for _ in range(12):
        a, b = torch.cuda.Event(True), torch.cuda.Event(True)
        a.record()
        for _ in range(5):
            _run(d)
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    return min(times)


@pytest.mark.parametrize("value", [5e6, -5e6, 1e9, -1e30])
@pytest.mark.parametrize("B", [1, 2, 4, 8])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("sparse", [False, True])
def test_masked_image(dev, value, B, cplx, sparse):
    w = W.small_random(seed=2, B=B, C=9, T=5, S=96, N=(6, 5, 23), K=3 if sparse else None,
                       complex_iq=cplx, sparse=sparse)
    d = to_dev(w, dev)
    d["offsets"].view(-1)[::7] = value
    d["weights"].view(-1)[::14] = float("nan")        # of slots that are passed over: not read
    import ffdas_amd
    ref = _run(d, algorithm=ffdas_amd.Algorithm.ALG1)
    assert ref.isfinite().all()
    assert rel_l2(_run(d).cpu().numpy(), ref.cpu().numpy()) < 1e-5


@pytest.mark.parametrize("B,cplx,K", [(1, False, 16), (2, False, 8), (8, True, 4)])
@pytest.mark.parametrize("value", [1e7, -1e30])
def test_masked_image_costs_no_more(dev, B, cplx, K, value):
    w = W.small_random(seed=2, B=B, C=96, T=K, S=1024, N=(256, 160), complex_iq=cplx)
    d = to_dev(w, dev)
    import torch
    z, x = torch.meshgrid(torch.linspace(60, 450, 256), torch.linspace(-300, 300, 160), indexing="ij")
    d["dstpos"] = torch.stack([x, 0 * x, z], -1).to(dev)
    d["srcpos"] = torch.stack([torch.linspace(-300, 300, 96), torch.zeros(96), torch.zeros(96)], -1).to(dev)
    o = d["offsets"] = (z + 0.02 * torch.arange(K).reshape(-1, 1, 1) * x).to(dev).contiguous()
    plain = _ms(d)
    o = o.clone()
    o[..., ::8, ::8] = value
    assert _ms(dict(d, offsets=o)) < 1.25 * plain
