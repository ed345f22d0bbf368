"""Complex FP32 frames of one and two slots, which take rounds of two, and of three, which do not (GPU),
against the FP64 oracle.
Tolerance: 1e-5 rel-L2, as every FP32 forward."""
import pytest

import oracle
from ffdas_amd import workloads as W
from tests.helpers import oracle_args, rel_l2, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [(13, 21), (5, 9, 6)])
@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("srcdir", [False, True])
@pytest.mark.parametrize("K", [1, 2, 3])
@pytest.mark.parametrize("B", [4, 8, 13, 16])
def test_image(dev, B, K, srcdir, sparse, N):
    import ffdas_amd
    w = W.small_random(seed=K, B=B, C=9, T=4 if sparse else K, S=64, N=N, K=K, complex_iq=True, srcdir=srcdir,
                       sparse=sparse)
    if sparse:
        w.sparse_indices.flat[::7] = -1
    d = to_dev(w, dev)
    si = d.pop("sparse_indices", None)
    geo = [d.pop(k) for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
    out = ffdas_amd.das_sparse(*geo, si, **d) if sparse else ffdas_amd.das(*geo, **d)
    args, kw = oracle_args(w)
    assert rel_l2(out.cpu().numpy(), oracle.das(*args, **kw)) < 1e-5
