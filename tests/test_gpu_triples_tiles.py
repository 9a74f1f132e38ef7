"""(T) at the sizes where the GEMM tiles of its products end: 16-column steps of the FP64 tile (its
width follows v), one and two column tiles, K halves of an odd number of 8-wide stages, and the
FP16x3 tiles with Y in 8 x 8 blocks and in plain rows, against ``oracle/triples_ref.py``.

Bars: FP64 sums of at most 2 (v + o) products of order one, summed over v^3 elements without
cancellation beyond that of E(T) itself: 1e-12 relative; FP16x3 products carry 2^-22 each and average
out over v^3 elements: 1e-8 relative."""
import pytest

from conftest import random_amplitudes
from oracle.triples_ref import t_tjl
from pycc_amd.synth import synthetic_df, DenseHamiltonian, dirac_eri

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# v: 16-column steps 1, 2, 4, 5, 7, 8 of one tile, then two tiles of 80; v + o padded to 8: 24, 40,
# 72, 80, 112 (o = 2, v = 104), 128 and 136
@pytest.mark.parametrize("no,nv", [(3, 16), (4, 31), (2, 64), (3, 73), (2, 104), (2, 120), (2, 129)])
def test_triples_at_tile_edges(no, nv):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pycc_amd
    print("triples tiles no=%d nv=%d" % (no, nv), flush=True)
    sd = synthetic_df(no, nv, seed=nv, t2max=0.1)
    H = DenseHamiltonian(sd.fock, dirac_eri(sd.B))
    t1, t2 = random_amplitudes(no, nv, nv, scale=0.1)
    ref = t_tjl(H.F, H.ERI, t1, t2, no)
    dp = pycc_amd.CCwfn(sd, no=no, precision='DP', verbose=False).triples_energy(t1, t2)
    assert abs(dp - ref) < 1e-12 * abs(ref), (dp, ref)
    x3 = pycc_amd.CCwfn(sd, no=no, precision='MIXED_F16X3', verbose=False).triples_energy(t1, t2)
    assert abs(x3 - dp) < 1e-8 * abs(dp), (x3, dp)
