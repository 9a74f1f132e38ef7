"""In the mixed precisions a contraction that fills the chip as a plain matrix product keeps that kernel, whatever
small contractions stand in the queue beside it: each kernel divides K by a rule of its own, and FP64 sums that are
rounded to FP32 or FP16 operands are to be divided by their shape alone. Read from the library's trace (CCX_TRACE),
which is decided once per process: hence the child process. 8 occupied and 256 virtual orbitals: t2_ijae G_be is
16384 x 256 x 256, 256 tiles, and -t2_imab Hm_mj is queued with it."""
import os
import subprocess
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = """
import torch, pycc_amd
from pycc_amd.synth import synthetic_df
sd = synthetic_df(8, 256, seed=1, naux=64)
cc = pycc_amd.CCwfn(sd, no=8, precision='MIXED', verbose=False)
g = torch.Generator(device='cuda').manual_seed(1)
t1 = 0.05 * torch.randn((8, 256), dtype=torch.float64, device='cuda', generator=g)
t2 = 0.05 * torch.randn((8, 8, 256, 256), dtype=torch.float64, device='cuda', generator=g)
t2 = t2 + t2.permute(1, 0, 3, 2)
r1, r2 = cc.residuals(cc.H.F, t1, t2.contiguous())
assert bool(torch.isfinite(r2).all())
"""


def test_a_plain_product_is_not_grouped():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    r = subprocess.run([sys.executable, "-c", PROGRAM], cwd=ROOT, env=dict(os.environ, CCX_TRACE="1"), capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    lines = r.stderr.splitlines()
    at = [i for i, l in enumerate(lines) if l.startswith("[ccx] ijae,be->ijab")]
    assert at
    for i in at:
        assert "-> plain" in lines[i + 1], lines[i:i + 2]
