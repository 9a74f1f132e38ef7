"""E(T) (pycc/cctriples.py:177-240) where the triples of a call fall into chunks of eight, the last one shorter: 20 triples
of four occupied orbitals at 190 virtual ones in FP64, 230 in MIXED_F16X3.

A triple's energy does not depend on its chunk, so ranges of i add up to the bits of one call, whatever their chunks;
the FP16x3 products keep E(T) to 1e-7 of the FP64 value (22-bit operands: 2^-22 = 2.4e-7 of a product, and the
sum over v^3 products averages it out)."""
import pytest

from conftest import random_amplitudes

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,nv", [("DP", 190), ("MIXED_F16X3", 230)])
def test_chunks_of_eight_triples(precision, nv):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import pycc_amd
    from pycc_amd.synth import synthetic_df
    sd = synthetic_df(4, nv, seed=nv, naux=64)
    t1, t2 = random_amplitudes(4, nv, 1, scale=0.01)
    t1, t2 = torch.tensor(t1, device="cuda"), torch.tensor(t2, device="cuda")
    cc = pycc_amd.CCwfn(sd, no=4, precision=precision, verbose=False)
    whole = cc.triples_energy(t1, t2)
    assert cc.triples_energy(t1, t2, i_chunk=1) == whole
    assert cc.triples_energy(t1, t2, i_chunk=3) == whole
    if precision != "DP":
        del cc
        ref = pycc_amd.CCwfn(sd, no=4, precision="DP", verbose=False).triples_energy(t1, t2)
        assert abs(whole - ref) < 1e-7 * abs(ref)
