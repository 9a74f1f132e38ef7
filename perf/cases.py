"""What this framework is used for, as cases that can be timed: coupled-cluster calls of one user's program
on one GPU, from a molecule of ten electrons to the largest systems of which several fit the card at once.

``listed()`` are the cases, ``draw(rng)`` gives more of the same ranges, ``prepare(case, seed)`` builds what a
program holds before the call (a wavefunction with its integrals on the GPU, amplitudes), ``run(state)`` is
one pass through the public entry points, ``work(case)`` is what that pass cannot do without, and
``exact(case, seed)`` is the same answer from plain torch in 64 bits.

The kinds of pass:

  solve      ``CCwfn.solve_cc`` from the MP1 amplitudes to loose thresholds (iterations, DIIS, energies)
  residual   ``CCwfn.residuals``: one amplitude residual, the step that the solve repeats
  lambda     ``cclambda.residuals``: one Lambda residual on a kept HBAR, the step that the Lambda solve repeats
  gradient   ``autograd.lagrangian`` and its backward at new amplitudes (residual, HBAR, vector-Jacobian product)
  jvp        ``CCwfn.jvp``: one Jacobian product on a kept HBAR, the step of a response or EOM solver
  triples    ``CCwfn.triples_energy``: E(T)

``precision`` is the framework's own option: DP, MIXED (FP32 products), MIXED_BF16X3, MIXED_F16X3.
"""
import math

import numpy as np
import torch

import pycc_amd
from pycc_amd import autograd

F64 = torch.float64


def listed():
    return [
        # Ten electrons in a double-zeta basis (the water example's o=5, v=19) with dense integrals: the whole
        # solve, every call of it far too small to fill the chip.
        {"name": "solve_o5_v19_dp", "kind": "solve", "o": 5, "v": 19, "precision": "DP", "dense": True},
        # A small molecule in a larger basis, odd extents.
        {"name": "residual_o9_v61_dp", "kind": "residual", "o": 9, "v": 61, "precision": "DP"},
        # The ordinary FP64 size (the o=16, v=128 of the synthetic Hamiltonians).
        {"name": "residual_o16_v128_dp", "kind": "residual", "o": 16, "v": 128, "precision": "DP"},
        # The FP32 form at odd extents: no leading dimension is a multiple of a vector.
        {"name": "residual_o19_v147_mixed", "kind": "residual", "o": 19, "v": 147, "precision": "MIXED"},
        # The large system in FP64 and in the split-product form that the benchmark runs.
        {"name": "residual_o32_v256_dp", "kind": "residual", "o": 32, "v": 256, "precision": "DP"},
        {"name": "residual_o32_v256_f16x3", "kind": "residual", "o": 32, "v": 256, "precision": "MIXED_F16X3"},
        # Lambda iterations: odd and ordinary in FP64, and large with split products.
        {"name": "lambda_o13_v101_dp", "kind": "lambda", "o": 13, "v": 101, "precision": "DP"},
        {"name": "lambda_o32_v256_f16x3", "kind": "lambda", "o": 32, "v": 256, "precision": "MIXED_F16X3"},
        # A gradient through autograd at new amplitudes: forward and backward.
        {"name": "gradient_o10_v77_dp", "kind": "gradient", "o": 10, "v": 77, "precision": "DP"},
        # A response solver's step.
        {"name": "jvp_o16_v128_dp", "kind": "jvp", "o": 16, "v": 128, "precision": "DP"},
        # E(T) in both precisions that it has, even and odd.
        {"name": "triples_o11_v107_dp", "kind": "triples", "o": 11, "v": 107, "precision": "DP"},
        {"name": "triples_o24_v176_f16x3", "kind": "triples", "o": 24, "v": 176, "precision": "MIXED_F16X3"},
    ]


# Drawn cases: kind -> (weight, precisions, largest v). v is spread over its logarithm, o follows v in the
# ratio that basis sets give (v/o from 4 to 12).
_DRAW = {
    "solve": (3, ("DP", "MIXED_F16X3"), 72),
    "residual": (6, ("DP", "DP", "MIXED_F16X3", "MIXED_F16X3", "MIXED", "MIXED_BF16X3"), 256),
    "lambda": (3, ("DP", "MIXED_F16X3"), 224),
    "gradient": (2, ("DP",), 144),
    "jvp": (2, ("DP",), 160),
    "triples": (3, ("DP", "MIXED_F16X3"), 160),
}


def draw(rng):
    kinds = sorted(_DRAW)
    kind = rng.choices(kinds, [_DRAW[k][0] for k in kinds])[0]
    _, precisions, vmax = _DRAW[kind]
    v = int(round(math.exp(rng.uniform(math.log(16), math.log(vmax)))))
    o = max(2, min(32, int(round(v / rng.uniform(4.0, 12.0)))))
    if kind == "triples":
        o = min(o, 16)
    case = {"kind": kind, "o": o, "v": v, "precision": rng.choice(precisions)}
    if kind == "solve" and o + v <= 48:
        case["dense"] = rng.random() < 0.5
    return case


# ---- inputs ----------------------------------------------------------------------------------------
class _DF:
    """A density-fitted Hamiltonian as ``CCwfn`` takes it: B (naux, nmo, nmo) and the Fock matrix."""


class _Dense:
    """A dense Hamiltonian: Dirac ERI <pq|rs> and the Fock matrix."""


def _randn(g, *shape):
    return torch.randn(*shape, dtype=F64, device="cuda", generator=g)


def _inputs(case, seed):
    """Orbital energies, B (naux = 2 nmo, decaying off the diagonal, scaled so that the largest MP1 doubles
    amplitude is 0.03), amplitudes near the MP1 ones and Lambda amplitudes / cotangents near theirs."""
    o, v = case["o"], case["v"]
    n = o + v
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    rng = np.random.default_rng(int(seed))
    eps = np.concatenate([np.sort(rng.uniform(-1.5, -0.4, o)), np.sort(rng.uniform(0.2, 3.0, v))])
    X = _randn(g, 2 * n, n, n)
    B = torch.triu(X) + torch.triu(X, 1).transpose(1, 2)
    i = torch.arange(n, device="cuda", dtype=F64)
    B *= torch.exp(-(i[:, None] - i[None, :]).abs() / n)
    e = torch.as_tensor(eps, device="cuda")
    eo, ev = e[:o], e[o:]
    flat = B[:, :o, o:].reshape(2 * n, o * v)
    iajb = (flat.t() @ flat).view(o, v, o, v)
    t2 = iajb.permute(0, 2, 1, 3) / (eo[:, None, None, None] + eo[:, None, None] - ev[:, None] - ev)
    scale = 0.03 / float(t2.abs().max())
    B *= math.sqrt(scale)
    t2 *= scale

    def near(x, by):
        x = x * (1.0 + by * _randn(g, *x.shape))
        return (0.5 * (x + x.permute(1, 0, 3, 2))).contiguous()

    t2 = near(t2, 0.1)
    t1 = 0.004 * _randn(g, o, v)
    l2 = near(2.0 * (2.0 * t2 - t2.transpose(2, 3)), 0.1)
    l1 = 2.0 * t1 + 0.002 * _randn(g, o, v)
    return {"eps": eps, "B": B.contiguous(), "t1": t1, "t2": t2, "l1": l1, "l2": l2}


def prepare(case, seed):
    x = _inputs(case, seed)
    if case.get("dense"):
        H = _Dense()
        n = case["o"] + case["v"]
        flat = x["B"].reshape(-1, n * n)
        H.F, H.ERI = np.diag(x["eps"]), (flat.t() @ flat).view(n, n, n, n).permute(0, 2, 1, 3).contiguous()
    else:
        H = _DF()
        H.fock, H.B = np.diag(x["eps"]), x["B"]
    cc = pycc_amd.CCwfn(H, no=case["o"], precision=case["precision"], verbose=False)
    s = {"kind": case["kind"], "cc": cc}
    if case["kind"] == "solve":
        s["t1"], s["t2"] = cc.t1.clone(), cc.t2.clone()
        return s
    s.update({k: x[k] for k in ("t1", "t2", "l1", "l2")})
    if case["kind"] == "lambda":
        cc.t1, cc.t2 = s["t1"], s["t2"]
        s["lam"] = pycc_amd.cclambda(cc, pycc_amd.cchbar(cc))
    return s


# Thresholds of the solve: a starting point for a tighter solver, or a scan's accuracy.
E_CONV, R_CONV = 1e-5, 1e-4


def run(s):
    cc, kind = s["cc"], s["kind"]
    if kind == "solve":
        cc.t1, cc.t2 = s["t1"].clone(), s["t2"].clone()
        e = cc.solve_cc(E_CONV, R_CONV)
        return {"e": e, "t1": cc.t1, "t2": cc.t2}
    if kind == "residual":
        r1, r2 = cc.residuals(cc.H.F, s["t1"], s["t2"])
        return {"r1": r1, "r2": r2}
    if kind == "lambda":
        r1, r2 = s["lam"].residuals(cc.H.F, s["t1"], s["t2"], s["l1"], s["l2"])
        return {"r1": r1, "r2": r2}
    if kind == "gradient":
        t1, t2 = s["t1"].clone().requires_grad_(), s["t2"].clone().requires_grad_()
        e = autograd.lagrangian(cc, t1, t2, s["l1"], s["l2"])
        g1, g2 = torch.autograd.grad(e, (t1, t2))
        return {"e": e.detach(), "g1": g1, "g2": g2}
    if kind == "jvp":
        j1, j2 = cc.jvp(s["t1"], s["t2"], s["l1"], s["l2"])
        return {"j1": j1, "j2": j2}
    return {"e": cc.triples_energy(s["t1"], s["t2"])}


# ---- what a pass cannot do without --------------------------------------------------------------------
def _contractions(o, v):
    """Multiply-adds x 2 of one amplitude residual with the ladder over symmetric and antisymmetric pairs."""
    pv, mv, po, mo = v * (v + 1) // 2, v * (v - 1) // 2, o * (o + 1) // 2, o * (o - 1) // 2
    ladder = 2.0 * po * (pv + o * v) * pv + 2.0 * mo * (mv + o * v) * mv
    ring = 12.0 * (o * v) ** 3
    holes = 4.0 * o ** 4 * v ** 2
    thin = 12.0 * o ** 2 * v ** 3 + 4.0 * o ** 2 * v ** 3 + 8.0 * o ** 3 * v ** 2 * 2
    return ladder, ring + holes + thin


def work(case):
    o, v, kind = case["o"], case["v"], case["kind"]
    ladder, rest = _contractions(o, v)
    word = 8.0 if case["precision"] == "DP" else 4.0
    amp = 8.0 * (o * v + o * o * v * v)
    # the integrals, each symmetry-unique element once: <ab|ef>, (me|af), two o^2 v^2 blocks, (mi|ne), (mi|nj)
    small = o * o * v * v * 1.0 + o ** 3 * v / 2.0 + o ** 4 / 8.0
    ints = word * (v ** 4 / 8.0 + o * v ** 3 / 2.0 + small)
    if kind == "triples":
        nt = o * (o + 1) * (o + 2) / 6.0
        return {"bytes": 8.0 * (o * v ** 3 / 2.0 + o ** 3 * v + o * o * v * v) + amp, "flops": 12.0 * nt * v ** 3 * (v + o)}
    if kind == "residual":
        return {"bytes": ints + 2 * amp, "flops": ladder + rest}
    if kind == "solve":
        return {"bytes": 8.0 * (ints / word) + 2 * amp, "flops": 6 * (ladder + rest)}   # about six iterations
    if kind in ("lambda", "jvp"):
        hbar = 8.0 * (2 * o * o * v * v + 2 * o ** 3 * v + o ** 4)
        return {"bytes": ints + hbar + 3 * amp, "flops": ladder + rest}
    return {"bytes": ints + 6 * amp, "flops": 2 * (ladder + rest) + rest}               # gradient: with HBAR


# ---- the same answers from plain torch in 64 bits --------------------------------------------------------
class _Plain:
    """Closed-shell CCSD equations over chemist blocks (pq|rs) = sum_Q B_Qpq B_Qrs."""

    def __init__(self, case, x):
        o, v = case["o"], case["v"]
        B = x["B"]
        self.o, self.v = o, v
        self.e = torch.as_tensor(x["eps"], device="cuda")
        self.Fo, self.Fv = torch.diag(self.e[:o]), torch.diag(self.e[o:])
        oo, ov, self.vv = B[:, :o, :o], B[:, :o, o:], B[:, o:, o:].contiguous()

        def block(p, q):
            n = p.shape[0]
            r = p.reshape(n, -1).t() @ q.reshape(n, -1)
            return r.view(p.shape[1], p.shape[2], q.shape[1], q.shape[2])

        self.oooo, self.ooov, self.oovv = block(oo, oo), block(oo, ov), block(oo, self.vv)
        self.ovov, self.ovvv = block(ov, ov), block(ov, self.vv)
        self.I = self.ovov.permute(0, 2, 1, 3).contiguous()             # <mn|ef>
        self.L = 2.0 * self.I - self.I.transpose(2, 3)                  # L_mnef
        self.Looov = 2.0 * self.ooov - self.ooov.permute(2, 1, 0, 3)    # [m,i,n,e] = 2(mi|ne) - (ni|me)
        self.Lovvv = 2.0 * self.ovvv - self.ovvv.permute(0, 3, 2, 1)    # [m,f,a,e] = 2(mf|ae) - (me|af)

    def mp1(self):
        eo, ev = self.e[:self.o], self.e[self.o:]
        return self.I / (eo[:, None, None, None] + eo[:, None, None] - ev[:, None] - ev)

    def ladder(self, tau):
        """sum_ef tau_ijef (ae|bf), a few a at a time."""
        o, v = self.o, self.v
        flat, out = tau.reshape(o * o, v * v), []
        q = self.vv.shape[0]
        for a in range(v):
            g = (self.vv[:, a, :].t() @ self.vv.reshape(q, v * v)).view(v, v, v)     # [e][b][f]
            out.append(flat @ g.transpose(1, 2).reshape(v * v, v))
        return torch.stack(out, 1).view(o, o, v, v)

    def residual(self, t1, t2):
        c = torch.einsum
        tt = c("ia,jb->ijab", t1, t1)
        tau, half = t2 + tt, t2 + 0.5 * tt
        u = 2.0 * t2 - t2.transpose(2, 3)
        Fme = c("nf,mnef->me", t1, self.L)
        Fae = self.Fv + c("mf,mfae->ae", t1, self.Lovvv) - c("mnaf,mnef->ae", half, self.L)
        Fmi = self.Fo + c("ne,mine->mi", t1, self.Looov) + c("inef,mnef->mi", half, self.L)
        Wmnij = self.oooo.permute(0, 2, 1, 3) + c("je,mine->mnij", t1, self.ooov) + c("ie,njme->mnij", t1, self.ooov)
        Wmnij = Wmnij + c("ijef,mnef->mnij", tau, self.I)
        mix = 0.5 * t2 + tt
        Wmbej = self.ovov.permute(0, 3, 1, 2) + c("jf,mebf->mbej", t1, self.ovvv) - c("nb,njme->mbej", t1, self.ooov)
        Wmbej = Wmbej - c("jnfb,mnef->mbej", mix, self.I) + 0.5 * c("njfb,mnef->mbej", t2, self.L)
        Wmbje = -self.oovv.permute(0, 2, 1, 3) - c("jf,mfbe->mbje", t1, self.ovvv) + c("nb,mjne->mbje", t1, self.ooov)
        Wmbje = Wmbje + c("jnfb,mnfe->mbje", mix, self.I)
        Z = c("mebf,ijef->mbij", self.ovvv, tau)
        r1 = c("ie,ae->ia", t1, Fae) - c("mi,ma->ia", Fmi, t1) + c("imae,me->ia", u, Fme)
        r1 = r1 + 2.0 * c("nf,nfia->ia", t1, self.ovov) - c("nf,niaf->ia", t1, self.oovv)
        r1 = r1 + c("mief,meaf->ia", u, self.ovvv) - c("mnae,mine->ia", t2, self.Looov)
        h = 0.5 * self.I + c("ijae,be->ijab", t2, Fae - 0.5 * c("mb,me->be", t1, Fme))
        h = h - c("imab,mj->ijab", t2, Fmi + 0.5 * c("je,me->mj", t1, Fme))
        h = h + 0.5 * c("mnab,mnij->ijab", tau, Wmnij) + 0.5 * self.ladder(tau) - c("ma,mbij->ijab", t1, Z)
        h = h + c("imae,mbej->ijab", u, Wmbej) + c("imae,mbje->ijab", t2, Wmbje) + c("mjae,mbie->ijab", t2, Wmbje)
        h = h - c("ma,ie,mejb->ijab", t1, t1, self.ovov) - c("mb,ie,mjae->ijab", t1, t1, self.oovv)
        h = h + c("ie,jbae->ijab", t1, self.ovvv) - c("ma,mijb->ijab", t1, self.ooov)
        return r1, h + h.permute(1, 0, 3, 2)

    def energy(self, t1, t2):
        return torch.sum((t2 + torch.einsum("ia,jb->ijab", t1, t1)) * self.L)

    def triples(self, t1, t2):
        """Sum over i >= j >= k of the closed-shell (T) terms, all a, b, c at once."""
        o, v = self.o, self.v
        ev = self.e[o:]
        D3 = ev[:, None, None] + ev[:, None] + ev
        total = torch.zeros((), dtype=F64, device="cuda")
        for i in range(o):
            for j in range(i + 1):
                for k in range(j + 1):
                    W = torch.zeros(v, v, v, dtype=F64, device="cuda")
                    # one term and its images under the six simultaneous permutations of (i, a), (j, b), (k, c)
                    for p, q, r, back in ((i, j, k, (0, 1, 2)), (i, k, j, (0, 2, 1)), (j, i, k, (1, 0, 2)),
                                          (j, k, i, (2, 0, 1)), (k, i, j, (1, 2, 0)), (k, j, i, (2, 1, 0))):
                        # x, y, z go with p, q, r: sum_d (px|yd) t_qr,dz ... written as two matrix products
                        X = (self.ovvv[p].reshape(v * v, v) @ t2[r, q].t()).view(v, v, v)
                        X = X - (t2[p].permute(1, 2, 0).reshape(v * v, o) @ self.ooov[:, q, r, :]).view(v, v, v)
                        W += X.permute(*back)
                    V = W + self.I[i, j][:, :, None] * t1[k] + self.I[i, k][:, None, :] * t1[j][:, None]
                    V = V + self.I[j, k] * t1[i][:, None, None]
                    R = 4.0 * W + W.permute(2, 0, 1) + W.permute(1, 2, 0)
                    R = R - 2.0 * (W.permute(0, 2, 1) + W.permute(1, 0, 2) + W.permute(2, 1, 0))
                    D = self.e[i] + self.e[j] + self.e[k] - D3
                    total = total + (2.0 - ((i == j) + (i == k) + (j == k))) * torch.sum(V * R / D)
        return total


def _sym(x):
    return x + x.permute(1, 0, 3, 2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        return None                  # to loose thresholds, the answer is the iteration's own
    x = _inputs(case, seed)
    p = _Plain(case, x)
    t1, t2, l1, l2 = x["t1"], x["t2"], x["l1"], x["l2"]
    if kind == "triples":
        return {"e": p.triples(t1, t2)} if case["o"] <= 24 else None
    if kind == "residual":
        r1, r2 = p.residual(t1, t2)
        return {"r1": r1, "r2": r2}
    if kind == "jvp":
        (_, _), (j1, j2) = torch.func.jvp(p.residual, (t1, t2), (l1, l2))
        return {"j1": j1, "j2": j2}
    t1.requires_grad_()
    t2.requires_grad_()
    r1, r2 = p.residual(t1, t2)
    e = p.energy(t1, t2) + torch.sum(l1 * r1) + 0.5 * torch.sum(l2 * r2)
    g1, g2 = torch.autograd.grad(e, (t1, t2))
    if kind == "lambda":
        return {"r1": g1, "r2": _sym(g2)}
    return {"e": e.detach(), "g1": g1, "g2": 0.5 * _sym(g2)}
