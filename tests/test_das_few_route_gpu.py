"""One to three frames on either side of the rule that gives them to the few-frames kernel (GPU): the same
image from both sides of the line as the FP64 oracle's, and the kernel that the rule names.
Tolerance: 1e-5 rel-L2, as every FP32 forward."""
import pytest

import oracle
from ffdas_amd import workloads as W
from tests.helpers import oracle_args, rel_l2, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,few", [((248, 250), True), ((256, 250), False), ((36, 40, 41), True), ((40, 40, 40), False)])
@pytest.mark.parametrize("B,cplx,sparse", [(1, False, False), (2, False, False), (3, False, False),
                                           (1, True, False), (1, False, True), (2, True, True)])
def test_either_kernel(dev, N, few, B, cplx, sparse):
    import torch
    import ffdas_amd
    from ffdas_amd.utils import profiling as P
    w = W.small_random(seed=B, B=B, C=3, T=2 if sparse else 1, S=64, N=N, K=1, complex_iq=cplx, sparse=sparse)
    d = to_dev(w, dev)
    geo = [d[k] for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
    P.reset()
    with P.profiled():
        out = (ffdas_amd.das_sparse(*geo, d["sparse_indices"], wavenum=w.wavenum) if sparse
               else ffdas_amd.das(*geo, wavenum=w.wavenum))
    torch.cuda.synchronize()
    assert (P.query("das_fwd_few")[1] > 0) == few and (P.query("das_fwd")[1] > 0) != few
    args, kw = oracle_args(w)
    assert rel_l2(out.cpu().numpy(), oracle.das(*args, **kw)) < 1e-5
