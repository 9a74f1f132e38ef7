"""Contractions (``ccx_contract``, pycc/device.py:64-86) whose two summed indices are each contiguous in another operand, so
that neither tile is read along a line, at both sides of the size from which these take 128 x 128 tiles only (512
tiles of 64 x 64), alone, as a batch and with a long sum that is split; and square products around 1000, whose split
counts the launch model decides.

The reference is torch's einsum in FP64 on the CPU. Tolerance: a sum of K products in any order is within (K + 4) u sum
|a||b| of the exact one (u the unit roundoff), and so is the reference."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _check(sub, ext, beta=-0.5):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pycc_amd
    lhs, out = sub.split("->")
    la, lb = lhs.split(",")
    g = torch.Generator().manual_seed(1)
    A, B, C = (torch.randn([ext[c] for c in l], dtype=torch.float64, generator=g) for l in (la, lb, out))
    K = 1
    for c in set(la) & set(lb) - set(out):
        K *= ext[c]
    ref = 0.75 * torch.einsum(sub, A, B) + beta * C
    mag = 0.75 * torch.einsum(sub, A.abs(), B.abs()) + abs(beta) * C.abs()
    got = pycc_amd.DeviceManager('GPU', 'DP').contract(sub, A.cuda(), B.cuda(), alpha=0.75, out=C.cuda(), beta=beta)
    assert float(((got.cpu() - ref).abs() - 2 * (K + 4) * 2.3e-16 * mag).max()) <= 0.0


# 1408 x 1408 (484 tiles), 1452 x 1452 (529); 65 x 41600, 64 x 41600; a batch of four 704 x 704
@pytest.mark.parametrize("sub,ext", [
    ("mbej,jnfb->menf", dict(m=11, e=128, n=11, f=128, b=61, j=11)),
    ("mbej,jnfb->menf", dict(m=11, e=132, n=11, f=132, b=61, j=11)),
    ("mbej,jnfb->menf", dict(m=11, e=132, n=11, f=132, b=200, j=11)),
    ("mbej,jnfb->menf", dict(m=13, e=5, n=64, f=650, b=9, j=8)),
    ("mbej,jnfb->menf", dict(m=16, e=4, n=64, f=650, b=9, j=8)),
    ("xmbej,xjnfb->xmenf", dict(x=5, m=11, e=64, n=11, f=64, b=31, j=11)),
])
def test_operands_without_a_common_line(sub, ext):
    _check(sub, ext)


@pytest.mark.parametrize("n", [700, 1000, 1024, 1280])
@pytest.mark.parametrize("sub", ["ak,kb->ab", "ka,bk->ab"])
def test_square_products_around_1000(sub, n):
    _check(sub, dict(a=n, b=n, k=n))
