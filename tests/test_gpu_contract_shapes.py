"""The contraction engine (``ccx_contract`` / ``ccx_contract_f32``, pycc/device.py:64-86) at the sizes where its
kernels change path: tile edges and remainders, extents of one, odd strides, long K with small outputs
(split K), three summed indices that do not fuse.

The reference is torch's einsum in FP64 on the CPU. Tolerance: a sum of K products in any order is
within (K + 4) u sum |a||b| of the exact one (u the unit roundoff), and so is the reference.
"""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def contract():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pycc_amd
    return pycc_amd.DeviceManager('GPU', 'DP').contract


def _check(contract, sub, ext, dtype, beta=0.0, seed=0):
    lhs, out = sub.split("->")
    la, lb = lhs.split(",")
    g = torch.Generator().manual_seed(seed)
    A, B, C = (torch.randn([ext[c] for c in l], dtype=torch.float64, generator=g).to(dtype) for l in (la, lb, out))
    K = 1
    for c in set(la) & set(lb) - set(out):
        K *= ext[c]
    ref = 0.75 * torch.einsum(sub, A.double(), B.double()) + beta * C.double()
    mag = 0.75 * torch.einsum(sub, A.double().abs(), B.double().abs()) + abs(beta) * C.double().abs()
    u = torch.finfo(dtype).eps
    got = C.cuda() if beta else None
    got = contract(sub, A.cuda(), B.cuda(), alpha=0.75, out=got, beta=beta)
    over = ((got.cpu().double() - ref).abs() - 2 * (K + 4) * u * mag).max()
    assert float(over) <= 0.0, (sub, ext, float(over))


# outputs of 1 .. 200 values with long K: the split-K sums and every grouping of the reduction
@pytest.mark.parametrize("m,n,k", [(1, 1, 9000), (13, 13, 30011), (5, 19, 4099), (67, 61, 2053), (1, 200, 777), (129, 65, 1500)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_split_k(contract, m, n, k, dtype, beta):
    _check(contract, "ak,bk->ab", {"a": m, "b": n, "k": k}, dtype, beta)


# tile edges (64 and 128) and remainders, odd and even extents: 16-byte loads with and without a late pair, every
# combination of contiguous index in A and B
@pytest.mark.parametrize("sub", ["ak,bk->ab", "ak,kb->ab", "ka,bk->ab", "ka,kb->ab", "ak,kb->ba"])
@pytest.mark.parametrize("m,n,k", [(64, 128, 32), (65, 129, 33), (127, 63, 17), (128, 191, 15), (257, 130, 2), (300, 301, 1),
                                   (1025, 1023, 47)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_tiles(contract, sub, m, n, k, dtype):
    _check(contract, sub, {"a": m, "b": n, "k": k}, dtype, beta=0.5)


# two-level rows and columns, two and three summed indices that do not fuse, inner extents under and over a k-tile
@pytest.mark.parametrize("sub", ["kaub,ukcd->abcd", "iumef,umefa->ia", "imef,efam->ia", "imef,fmea->ia", "mnab,nmba->a",
                                 "xmey,mfxe->fy", "mief,meaf->ia", "jnfb,mnef->mbej"])
@pytest.mark.parametrize("occ,vir", [(3, 17), (5, 16), (17, 31), (2, 40)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_compound_indices(contract, sub, occ, vir, dtype):
    ext = {c: (vir if c in "abcdefg" else occ) for c in sub if c.isalpha()}
    _check(contract, sub, ext, dtype)


def test_rows_more_than_4_gib_apart(contract):
    """Rows of A 2 GiB apart: lane offsets past 32 bits."""
    step, rows, k, n = 1 << 28, 3, 37, 21
    buf = torch.empty((rows - 1) * step + k, dtype=torch.float64, device="cuda")
    A = torch.as_strided(buf, (rows, k), (step, 1))
    g = torch.Generator().manual_seed(1)
    a, b = torch.randn(rows, k, dtype=torch.float64, generator=g), torch.randn(k, n, dtype=torch.float64, generator=g)
    A.copy_(a)
    for sub, B in (("ak,kb->ab", b), ("ak,bk->ab", b.t().contiguous())):
        out = contract(sub, A, B.cuda()).cpu()
        assert float((out - a @ b).abs().max()) <= 2 * (k + 4) * 2.2e-16 * float((a.abs() @ b.abs()).max())


# every count of 16-row and 16-column blocks that a 64 x 64 tile can hold, alone and after a whole tile
@pytest.mark.parametrize("m", [7, 17, 40, 64, 78, 91, 107])
@pytest.mark.parametrize("n", [13, 30, 45, 61, 80, 100, 115])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_blocks_of_a_tile(contract, m, n, dtype):
    _check(contract, "ak,kb->ab", {"a": m, "b": n, "k": 53}, dtype, beta=0.5)


# aligned matrices of many tiles whose last tile row is short
@pytest.mark.parametrize("sub", ["ak,kb->ab", "ak,bk->ab", "ka,kb->ab"])
@pytest.mark.parametrize("m", [514, 528, 612, 640])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_short_last_tile_row(contract, sub, m, dtype):
    _check(contract, sub, {"a": m, "b": 8192, "k": 64}, dtype, beta=0.5)
