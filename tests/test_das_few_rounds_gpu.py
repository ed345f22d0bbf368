"""The forward for few frames where the slots fill whole rounds of 8 or of 16, or leave a remainder, against
the FP64 oracle (GPU).  Tolerance: 1e-5 rel-L2, as every FP32 forward."""
import pytest

import oracle
from ffdas_amd import workloads as W
from tests.helpers import oracle_args, rel_l2, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [15, 17, 18, 19, 20, 24, 31, 32, 35, 36, 40])
@pytest.mark.parametrize("cone", [False, True])
def test_rounds(dev, K, cone):
    import ffdas_amd
    w = W.small_random(seed=K, B=1, C=7, T=K, S=83, N=(13, 11), K=K, srcdir=cone)
    d = to_dev(w, dev)
    args, kw = oracle_args(w)
    geo = [d.pop(k) for k in ("x", "srcpos", "dstpos", "offsets", "weights")]
    assert rel_l2(ffdas_amd.das(*geo, **d).cpu().numpy(), oracle.das(*args, **kw)) < 1e-5
