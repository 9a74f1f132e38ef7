"""The residual, the Lambda residual and the JVP at both sides of the sizes where their launches are
arranged differently: (ov)^2 = 2^19 and 2^22 (the number of partial sums of a doubles residual), 2^20
(partial sums of W) and ov = 1024 (matrix-vector terms with launches of their own), against the oracles
of ``oracle/ccsd_ref.py`` and ``oracle/lambda_ref.py``.

Bar: FP64 sums of up to v^3 (2.7e5) products round to sqrt(2.7e5) 2^-53 = 6e-14 of their terms, a handful of
such sums to a residual element, and some hundred terms' cancellation: 1e-11 of the largest element (or of 1)."""
import numpy as np
import pytest

from conftest import random_amplitudes
from oracle.ccsd_ref import OracleCCSD
from oracle.lambda_ref import OracleHBAR, OracleLambda, ccsd_jacobian
from pycc_amd.synth import synthetic_df, DenseHamiltonian, dirac_eri

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _dev(x):
    return torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda")


def _rel(a, b):
    return float(np.abs(a.detach().cpu().numpy() - b).max() / max(1.0, np.abs(b).max()))


def _sym2(x):
    return 0.5 * (x + x.transpose(1, 0, 3, 2))


def _setup(no, nv):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pycc_amd
    print("queue routes no=%d nv=%d" % (no, nv), flush=True)
    sd = synthetic_df(no, nv, seed=no + nv, t2max=0.05)
    H = DenseHamiltonian(sd.fock, dirac_eri(sd.B))
    t1, t2 = random_amplitudes(no, nv, nv, scale=0.05)
    return H, pycc_amd.CCwfn(H, no=no, precision='DP', verbose=False), OracleCCSD(H, no), t1, _sym2(t2)


# (ov)^2: 518400, 541696 (2^19 = 524288); 2^20 with ov = 1024, 1081600; 2^22, 4322241
@pytest.mark.parametrize("no,nv", [(16, 45), (16, 46), (16, 64), (16, 65), (32, 64), (33, 63)])
def test_residual_either_side_of_the_routes(no, nv):
    H, cc, ref, t1, t2 = _setup(no, nv)
    r1, r2 = ref.residuals(H.F, t1, t2)
    g1, g2 = cc.residuals(H.F, t1, t2)
    assert _rel(g1, r1) < 1e-11 and _rel(g2, r2) < 1e-11


@pytest.mark.parametrize("no,nv", [(16, 45), (16, 46), (16, 65)])
def test_derivatives_either_side_of_the_routes(no, nv):
    H, cc, ref, t1, t2 = _setup(no, nv)
    l1, l2 = random_amplitudes(no, nv, nv + 2, scale=0.5)
    x1, x2 = random_amplitudes(no, nv, nv + 5, scale=1.0)
    l2 = _sym2(l2)
    oh = OracleHBAR(ref, t1, t2)
    r1, r2 = OracleLambda(ref, oh).residuals_with(oh, t2, l1, l2)
    cc._hbar_for(cc.H.F, _dev(t1), _dev(t2), True)
    g1, g2 = cc._lambda_residual(_dev(l1), _dev(l2), with_source=True)
    assert _rel(g1, r1) < 1e-11 and _rel(g2, r2) < 1e-11
    j1, j2 = ccsd_jacobian(ref, oh, x1, x2, t2=t2)
    g1, g2 = cc.jvp(_dev(t1), _dev(t2), _dev(x1), _dev(x2), store_vvvv=True)
    assert _rel(g1, j1) < 1e-11 and _rel(g2, j2 + j2.transpose(1, 0, 3, 2)) < 1e-11
