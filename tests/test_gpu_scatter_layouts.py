"""GPU test of the Lambda residual in a MIXED_F16X3 context at odd extents, against a DP context: at o=17, v=251 the
split products are scattered into outputs whose contiguous index is the products' own or another one, with
ragged 64 x 64 tiles (``pycc/cclambda.py:345-369, :468-496``).

Tolerance: each split product carries about 2^-22 relative error, the bar is 1e-6 relative (norm).
"""
import numpy as np
import pytest

from conftest import random_amplitudes
from pycc_amd.synth import synthetic_df

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("no,nv,seed", [(17, 251, 43)])
def test_lambda_residual_odd_extents(no, nv, seed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pycc_amd
    print("mixed Lambda residual vs DP no=%d nv=%d" % (no, nv), flush=True)

    def dev(x):
        return torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda")

    sd = synthetic_df(no, nv, seed=seed)
    t1, t2 = random_amplitudes(no, nv, seed + 1, scale=0.02)
    t1, t2 = dev(t1), dev(0.5 * (t2 + t2.transpose(1, 0, 3, 2)))
    rng = np.random.default_rng(seed)
    l1 = dev(rng.standard_normal((no, nv)) * 0.05)
    l2 = rng.standard_normal((no, no, nv, nv)) * 0.02
    l2 = dev(l2 + l2.transpose(1, 0, 3, 2))
    r = {}
    for precision in ('DP', 'MIXED_F16X3'):
        cc = pycc_amd.CCwfn(sd, no=no, precision=precision, verbose=False)
        cc._hbar_for(cc.H.F, t1, t2)
        r[precision] = cc._lambda_residual(l1, l2, with_source=True)
        torch.cuda.synchronize()
    for mixed, dp in zip(r['MIXED_F16X3'], r['DP']):
        assert float(torch.linalg.vector_norm(mixed - dp) / torch.linalg.vector_norm(dp)) < 1e-6
