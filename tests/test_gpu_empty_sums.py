"""Sums over nothing: contractions with a summed index of extent 0 (``ccx_contract`` / ``ccx_contract_f32``,
pycc/device.py:64-86), which give beta C, and CCSD with one virtual orbital (HF in a minimal basis), whose
antisymmetric ladder sums over no pair e < f.

An empty sum leaves nothing to round: the bar of the contractions is equality. The residuals, Lambda residuals and JVPs
of three orbitals are sums of some hundred terms of at most ten times the result, each rounded to 1e-16 of its size: 1e-12 of the
largest element (or of 1) in FP64; the FP32 products of 'MIXED' are a few of them, rounded to 6e-8: 1e-6."""
import ctypes

import numpy as np
import pytest

from conftest import random_amplitudes
from oracle.ccsd_ref import OracleCCSD
from oracle.lambda_ref import OracleHBAR, OracleLambda, ccsd_jacobian
from pycc_amd.synth import synthetic_df, DenseHamiltonian, dirac_eri

torch = pytest.importorskip("torch")

SUMS = [("ik,kj->ij", dict(i=5, j=7, k=0)), ("ki,kj->ij", dict(i=130, j=67, k=0)), ("ik,jk->ji", dict(i=1, j=3, k=0)),
        ("bik,bkj->bij", dict(b=4, i=5, j=6, k=0)), ("ikl,lkj->ij", dict(i=5, j=6, k=3, l=0)),
        ("iklm,mlkj->ij", dict(i=5, j=6, k=3, l=0, m=2)), ("iklm,mlkj->ij", dict(i=5, j=6, k=0, l=0, m=0)),
        ("k,k->", dict(k=0)), ("iakb,kjcd->iajcbd", dict(i=2, a=3, k=0, b=2, j=3, c=2, d=3))]


def _i64(x):
    return (ctypes.c_int64 * max(1, len(x)))(*x)


def _strides(shape):
    s, out = 1, []
    for n in reversed(shape):
        out.append(s)
        s *= n
    return out[::-1]


def _call(lib, sub, ext, alpha, beta, ptr, pc, dtype):
    lhs, out = sub.split("->")
    la, lb = lhs.split(",")
    args = []
    for lab, p in ((la, ptr), (lb, ptr), (out, pc)):
        shape = [ext[c] for c in lab]
        args.append((ctypes.c_void_p(p), _i64(shape), _i64(_strides(shape))))
    fn = lib.ccx_contract if dtype == torch.float64 else lib.ccx_contract_f32
    return fn(sub.encode(), alpha, *args[0], *args[1], beta, *args[2], None)


def _library():
    from pycc_amd import _lib
    try:
        return _lib.load()
    except Exception as e:
        pytest.skip("library not built: %s" % e)


@pytest.mark.parametrize("sub,ext", SUMS)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_an_empty_sum_is_accepted(sub, ext, dtype):
    """Without a GPU the call comes as far as its launch (CCX_ERR_HIP): it is not refused on the way."""
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    buf = (ctypes.c_double * 64)()
    p = ctypes.addressof(buf)
    assert _call(_library(), sub, ext, 0.75, 0.5, p, p, dtype) == -2


@pytest.mark.gpu
@pytest.mark.parametrize("sub,ext", SUMS)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_an_empty_sum_is_beta_c(sub, ext, dtype, beta):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    out = [ext[c] for c in sub.split("->")[1]]
    C = torch.randn(out, dtype=dtype, device="cuda") if beta else torch.full(out, float("nan"), dtype=dtype, device="cuda")
    want = beta * C if beta else torch.zeros_like(C)
    some = torch.ones(8, dtype=dtype, device="cuda")
    assert _call(_library(), sub, ext, 0.75, beta, some.data_ptr(), C.data_ptr(), dtype) == 0
    torch.cuda.synchronize()
    assert torch.equal(C, want)


def _sym2(x):
    return 0.5 * (x + x.transpose(1, 0, 3, 2))


def _dev(x):
    return torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda")


def _err(a, b):
    return float(np.abs(a.cpu().numpy() - b).max() / max(1.0, np.abs(b).max()))


def _one_virtual(no, precision):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pycc_amd
    sd = synthetic_df(no, 1, seed=no, t2max=0.05)
    H = DenseHamiltonian(sd.fock, dirac_eri(sd.B))
    t1, t2 = random_amplitudes(no, 1, no + 1, scale=0.05)
    return H, pycc_amd.CCwfn(H, no=no, precision=precision, verbose=False), OracleCCSD(H, no), t1, _sym2(t2)


@pytest.mark.gpu
@pytest.mark.parametrize("no", [1, 2, 3, 5])
@pytest.mark.parametrize("precision,tol", [("DP", 1e-12), ("MIXED", 1e-6)])
def test_residual_with_one_virtual(no, precision, tol):
    H, cc, ref, t1, t2 = _one_virtual(no, precision)
    r1, r2 = ref.residuals(H.F, t1, t2)
    g1, g2 = cc.residuals(H.F, t1, t2)
    assert _err(g1, r1) < tol and _err(g2, r2) < tol


@pytest.mark.gpu
@pytest.mark.parametrize("no", [1, 2, 3, 5])
@pytest.mark.parametrize("stored", [False, True])
def test_derivatives_with_one_virtual(no, stored):
    H, cc, ref, t1, t2 = _one_virtual(no, "DP")
    l1, l2 = random_amplitudes(no, 1, 7, scale=0.5)
    x1, x2 = random_amplitudes(no, 1, 8, scale=1.0)
    l2 = _sym2(l2)
    oh = OracleHBAR(ref, t1, t2)
    r1, r2 = OracleLambda(ref, oh).residuals_with(oh, t2, l1, l2)
    cc._hbar_for(cc.H.F, _dev(t1), _dev(t2), stored)
    g1, g2 = cc._lambda_residual(_dev(l1), _dev(l2), with_source=True)
    assert _err(g1, r1) < 1e-12 and _err(g2, r2) < 1e-12
    j1, j2 = ccsd_jacobian(ref, oh, x1, x2, t2=t2)
    g1, g2 = cc.jvp(_dev(t1), _dev(t2), _dev(x1), _dev(x2), store_vvvv=stored)
    assert _err(g1, j1) < 1e-12 and _err(g2, j2 + j2.transpose(1, 0, 3, 2)) < 1e-12


def test_empty_indices_of_any_strides():
    """Several empty indices whose strides do not nest: an empty output is nothing to do, an empty sum comes as far as its
    launch."""
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    lib, buf = _library(), (ctypes.c_double * 64)()
    p = ctypes.c_void_p(ctypes.addressof(buf))

    def call(sub, *views):
        args = [x for shape, strides in views for x in (p, _i64(shape), _i64(strides))]
        return lib.ccx_contract(sub.encode(), 1.0, *args[:6], 0.5, *args[6:], None)

    assert call("ab,ba->ab", ((0, 0), (5, 1)), ((0, 0), (3, 1)), ((0, 0), (2, 1))) == 0
    assert call("xab,xba->xab", ((3, 0, 0), (9, 5, 1)), ((3, 0, 0), (8, 3, 1)), ((3, 0, 0), (7, 2, 1))) == 0
    assert call("abcd,d->cab", ((0, 0, 0, 3), (9, 5, 3, 1)), ((3,), (1,)), ((0, 0, 0), (7, 2, 1))) == 0
    assert call("abc,cba->", ((0, 0, 0), (5, 3, 1)), ((0, 0, 0), (7, 2, 1)), ((), ())) == -2
    assert call("abcd,dcba->", ((0, 0, 0, 0), (9, 5, 3, 1)), ((0, 0, 0, 0), (11, 7, 2, 1)), ((), ())) == -2
