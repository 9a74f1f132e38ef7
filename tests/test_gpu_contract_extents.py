"""Contractions (``ccx_contract`` / ``ccx_contract_f32``, pycc/device.py:64-86) at the ends of the index range: sums
and outputs whose extent nears or passes 2^31. Operands are overlapping views of small buffers of whole numbers, so
that every sum is exact and the bar is equality."""
import ctypes

import pytest

torch = pytest.importorskip("torch")


def _i64(x):
    return (ctypes.c_int64 * max(1, len(x)))(*x)


def _library():
    from pycc_amd import _lib
    try:
        return _lib.load()
    except Exception as e:
        pytest.skip("library not built: %s" % e)


def _call(sub, dtype, views, beta=0.0):
    """views: (pointer, shape, strides) of A, B, C."""
    a, b, c = [(ctypes.c_void_p(p), _i64(shape), _i64(strides)) for p, shape, strides in views]
    lib = _library()
    fn = lib.ccx_contract if dtype == torch.float64 else lib.ccx_contract_f32
    return fn(sub.encode(), 1.0, *a, *b, beta, *c, None)


def _whole(n, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-1, 2, (n,), device="cuda", generator=g).to(dtype)


THREE = dict(shape=(1290, 1291, 1292), sa=(3, 5, 7), sb=(1, 4, 2))   # 2^31 + 4.2e6 products


def test_three_summed_indices_past_2_31_are_accepted():
    """Without a GPU the call comes as far as its launch (CCX_ERR_HIP): it is not refused on the way."""
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    buf = (ctypes.c_double * 64)()
    p = ctypes.addressof(buf)
    for dtype in (torch.float64, torch.float32):
        k, l, m = THREE["shape"]
        assert _call("klm,mlk->", dtype, [(p, (k, l, m), THREE["sa"]), (p, (m, l, k), THREE["sb"][::-1]), (p, (), ())]) == -2


@pytest.mark.gpu
def test_three_summed_indices_past_2_31():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    k, l, m = THREE["shape"]
    sa, sb = THREE["sa"], THREE["sb"]
    A, B = _whole(3 * k + 5 * l + 7 * m, torch.float64, 1), _whole(k + 4 * l + 2 * m, torch.float64, 2)
    C = torch.full((1,), 3.0, dtype=torch.float64, device="cuda")
    assert _call("klm,mlk->", torch.float64, [(A.data_ptr(), (k, l, m), sa), (B.data_ptr(), (m, l, k), sb[::-1]),
                                              (C.data_ptr(), (), ())], beta=2.0) == 0
    want = 6.0
    for i in range(k):
        want += float((torch.as_strided(A, (l, m), sa[1:], i * sa[0]) * torch.as_strided(B, (l, m), sb[1:], i * sb[0])).sum())
    assert float(C) == want


# one row of outputs as wide as an index goes, B row-fast and k-fast; past 2^30 columns a launch of 64-wide tiles has
# more threads than its x extent holds
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,n", [(torch.float32, (1 << 31) - 1), (torch.float64, (1 << 30) + 77)])
@pytest.mark.parametrize("step", [1, 5])
def test_one_row_of_very_many_columns(dtype, n, step):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    K = 3
    B = _whole(n + step * K, dtype, 3)
    a = torch.tensor([1.0, -2.0, 3.0], dtype=dtype, device="cuda")
    C = torch.empty(n, dtype=dtype, device="cuda")
    assert _call("k,kn->n", dtype, [(a.data_ptr(), (K,), (1,)), (B.data_ptr(), (K, n), (step, 1)), (C.data_ptr(), (n,), (1,))]) == 0
    for k, x in enumerate((1.0, -2.0, 3.0)):
        C.sub_(B[k * step:k * step + n], alpha=x)
    assert int(torch.count_nonzero(C)) == 0


# a sum as long as an index goes: of equal ones (no stride), and of a buffer that holds ones only at both ends
@pytest.mark.gpu
def test_a_sum_of_very_many_products():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    k = (1 << 31) - 1
    one = torch.ones(1, dtype=torch.float64, device="cuda")
    out = torch.empty(1, dtype=torch.float64, device="cuda")
    assert _call("k,k->", torch.float64, [(one.data_ptr(), (k,), (0,))] * 2 + [(out.data_ptr(), (), ())]) == 0
    assert float(out) == k
    x = torch.zeros(k, dtype=torch.float32, device="cuda")
    x[:3] = 1.0
    x[-20:] = 2.0
    out = torch.empty(1, dtype=torch.float32, device="cuda")
    assert _call("k,k->", torch.float32, [(x.data_ptr(), (k,), (1,))] * 2 + [(out.data_ptr(), (), ())]) == 0
    assert float(out) == 3.0 + 20 * 4.0
