"""GPU tests of the FP16x3 split GEMM (ccx_gemm_f16x3) where its last row of 256-row tiles is short: up to 32 and up
to 128 rows are computed by loops of their own, more of them as a whole tile.

A row of the product does not depend on the rows beside it, so the first M rows of a product whose A ends in zero
rows (whole tiles, the same scales and split of K) are the same bits. Against the FP64 product the
bar is that of the other split GEMM tests: 1e-6 of the largest |A| |B|, four FP32 roundings.
"""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mgr():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pycc_amd
    return pycc_amd.DeviceManager('GPU', 'MIXED_F16X3')


@pytest.mark.parametrize("N", [520, 8200])            # 256 and 320 columns per tile
@pytest.mark.parametrize("M", [257, 272, 288, 289, 384, 385, 528, 1040])
@pytest.mark.parametrize("K", [40, 1100])
def test_short_last_tile_row(mgr, M, N, K):
    print("short last row", M, N, K, flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    whole = (M + 255) // 256 * 256
    A = torch.zeros(whole, K, device="cuda")
    A[:M] = torch.randn(M, K, device="cuda", generator=g)
    B = torch.randn(K, N, device="cuda", generator=g)
    C0 = torch.randn(whole, N, device="cuda", generator=g)
    guard = torch.full((whole, N), 7.0, device="cuda")
    guard[:M] = C0[:M]
    C = mgr.contract.matmul_f16x3(A[:M], B, out=guard[:M], alpha=0.5, beta=2.0)
    ref = mgr.contract.matmul_f16x3(A, B, out=C0.clone(), alpha=0.5, beta=2.0)[:M]
    assert torch.equal(C, ref)
    assert torch.all(guard[M:] == 7.0)                 # nothing is written past row M
    exact = 0.5 * (A[:M].double() @ B.double()) + 2.0 * C0[:M].double()
    scale = 0.5 * float((A[:M].abs().double() @ B.abs().double()).max())
    assert float((C.double() - exact).abs().max()) < 1e-6 * scale
