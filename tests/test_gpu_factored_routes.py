"""The Lambda residual and the JVP on the factored HBAR (the default form), and the residuals of the mixed precisions, at
both sides of the sizes where their launches are arranged differently: (ov)^2 = 2^19 and 2^22 (the number of partial
sums; above 2^22 temporaries are shared and every term is added into one array), 2^20 (partial sums of W), against the
oracles of ``oracle/ccsd_ref.py`` and ``oracle/lambda_ref.py``.

Bars: FP64 as in the tests of the stored form, sums of up to v^3 (2.7e5) products that round to 6e-14 of their terms and some
hundred terms' cancellation: 1e-11 of the largest element (or of 1). The mixed precisions' residuals to the bars of
their parity tests, 1e-5 (FP32), 3e-4 (BF16x3 ladder), 3e-5 (FP16x3) of the largest element."""
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


def _ham(no, nv):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print("factored routes no=%d nv=%d" % (no, nv), flush=True)
    sd = synthetic_df(no, nv, seed=no + nv, t2max=0.05)
    H = DenseHamiltonian(sd.fock, dirac_eri(sd.B))
    t1, t2 = random_amplitudes(no, nv, nv, scale=0.05)
    return H, OracleCCSD(H, no), t1, _sym2(t2)


# (ov)^2: 518400, 541696 (2^19 = 524288); 1081600 (2^20); 4322241 (2^22)
SIZES = [(16, 45), (16, 46), (16, 65), (33, 63)]


@pytest.mark.parametrize("no,nv", SIZES)
def test_derivatives_on_the_factored_hbar(no, nv):
    H, ref, t1, t2 = _ham(no, nv)
    import pycc_amd
    cc = pycc_amd.CCwfn(H, no=no, precision='DP', verbose=False)
    l1, l2 = random_amplitudes(no, nv, nv + 2, scale=0.5)
    x1, x2 = random_amplitudes(no, nv, nv + 5, scale=1.0)
    l2 = _sym2(l2)
    oh = OracleHBAR(ref, t1, t2)
    cc._hbar_for(cc.H.F, _dev(t1), _dev(t2), False)
    r1, r2 = OracleLambda(ref, oh).residuals_with(oh, t2, l1, l2)
    g1, g2 = cc._lambda_residual(_dev(l1), _dev(l2), with_source=True)
    assert _rel(g1, r1) < 1e-11 and _rel(g2, r2) < 1e-11
    j1, j2 = ccsd_jacobian(ref, oh, x1, x2, t2=t2)
    g1, g2 = cc.jvp(_dev(t1), _dev(t2), _dev(x1), _dev(x2))
    assert _rel(g1, j1) < 1e-11 and _rel(g2, j2 + j2.transpose(1, 0, 3, 2)) < 1e-11


@pytest.mark.parametrize("no,nv", SIZES)
def test_mixed_residuals_either_side_of_the_routes(no, nv):
    H, ref, t1, t2 = _ham(no, nv)
    import pycc_amd
    r1, r2 = ref.residuals(H.F, t1, t2)
    for precision, tol in (("MIXED", 1e-5), ("MIXED_BF16X3", 3e-4), ("MIXED_F16X3", 3e-5)):
        cc = pycc_amd.CCwfn(H, no=no, precision=precision, verbose=False)
        g1, g2 = cc.residuals(H.F, t1, t2)
        assert _rel(g1, r1) < tol and _rel(g2, r2) < tol, precision
