"""Work that a user of this framework has it do, as cases to be timed.

Every case goes through the public entry points: the vector function and its
backward pass on device tensors (dalton_amd.autograd), and CCContext, CCBatch
and df_factor_ao on host arrays, as a driver program calls them.  Systems are
synthetic density-fitted closed-shell systems (Gaussian factor at half the
scale at which the CCSD iteration of such a system stops converging), with o
occupied and v virtual orbitals and naux auxiliary functions; sizes run from a
water molecule in a double-zeta basis to 32 occupied and 256 virtual orbitals.

  listed()   the cases        draw(rng)  one more of the same ranges
  prepare    inputs, contexts and amplitudes a program holds before the call
  run        one pass          exact      the same values in plain float64
  work       bytes and flops a pass cannot do without
"""
from __future__ import annotations

import math

import numpy as np
import torch

import dalton_amd as d
from dalton_amd.autograd import ccsd_residual

PRECISION = {"fp64": d.FP64, "mixed": d.MIXED, "fp32": d.FP32}
DEV = "cuda"


def listed():
    return [
        # one vector function of a water-sized molecule: the smallest call, launches and latency
        {"name": "rhs_fp64_o5_v19", "kind": "rhs", "prec": "fp64", "o": 5, "v": 19, "naux": 110},
        # the whole CCSD(T) energy of that molecule, from the MP2 guess to E4 and E5
        {"name": "ccsdt_fp64_o5_v19", "kind": "ccsdt", "prec": "fp64", "o": 5, "v": 19, "naux": 110},
        # a mid-sized molecule with odd dimensions, reference precision
        {"name": "rhs_fp64_o21_v170", "kind": "rhs", "prec": "fp64", "o": 21, "v": 170, "naux": 683},
        # the same in the split-product precision, smaller and odd in every dimension
        {"name": "rhs_mixed_o13_v117", "kind": "rhs", "prec": "mixed", "o": 13, "v": 117, "naux": 469},
        # the largest vector function: the size the left transformation and multipliers are quoted at
        {"name": "rhs_mixed_o32_v256", "kind": "rhs", "prec": "mixed", "o": 32, "v": 256, "naux": 1024},
        # a converged ground state in mixed precision (split products first, float64 at the end)
        {"name": "solve_mixed_o16_v128", "kind": "solve", "prec": "mixed", "o": 16, "v": 128, "naux": 512},
        # vector function and its left transformation (forward and backward), both precisions
        {"name": "grad_fp64_o11_v93", "kind": "grad", "prec": "fp64", "o": 11, "v": 93, "naux": 371},
        {"name": "grad_mixed_o24_v192", "kind": "grad", "prec": "mixed", "o": 24, "v": 192, "naux": 768},
        # (T): the full triple list of a small system, and a slice of a large one's
        {"name": "pt_fp64_o12_v101", "kind": "pt", "prec": "fp64", "o": 12, "v": 101, "naux": 404, "count": 0, "stride": 1},
        {"name": "pt_mixed_o32_v256", "kind": "pt", "prec": "mixed", "o": 32, "v": 256, "naux": 1024, "count": 64,
         "stride": 89},
        # uneven small systems converged together
        {"name": "batch_fp64", "kind": "batch", "prec": "fp64", "shapes": "5x40 5x57 7x61 8x90 10x83 12x110"},
        # the front end: AO integrals on the host to a density-fitting factor on the host
        {"name": "ao_factor_n90", "kind": "ao", "nbas": 90, "nmo": 90, "rank": 520},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: kind, precision and sizes over the listed ranges, cut so
    that it costs no more than the largest listed cases."""
    kind = rng.choice(["rhs", "rhs", "rhs", "grad", "grad", "solve", "pt", "pt", "ccsdt", "batch", "ao"])
    if kind == "ao":
        nbas = _log_int(rng, 20, 90)
        return {"kind": "ao", "nbas": nbas, "nmo": nbas - rng.randint(0, nbas // 8), "rank": rng.randint(3, 6) * nbas}
    if kind == "batch":
        shapes = []
        for _ in range(rng.randint(2, 6)):
            o = rng.randint(5, 11)
            shapes.append("%dx%d" % (o, rng.randint(8 * o, 10 * o)))
        return {"kind": "batch", "prec": rng.choice(["fp64", "mixed"]), "shapes": " ".join(shapes)}
    precs = {"rhs": ["fp64", "mixed", "mixed", "fp32"], "grad": ["fp64", "mixed"], "solve": ["fp64", "mixed"],
             "pt": ["fp64", "mixed"], "ccsdt": ["fp64", "mixed"]}[kind]
    prec = rng.choice(precs)
    # flops of one pass, at most what about a tenth of a second allows
    most = {"fp64": 3e12, "mixed": 12e12, "fp32": 5e12}[prec]
    top = {"rhs": 32, "grad": 24, "solve": 16, "pt": 32, "ccsdt": 9}[kind]
    o = _log_int(rng, 4, top)
    v = min(256, max(15, int(o * rng.uniform(3.6, 11.0))))
    while True:
        case = {"kind": kind, "prec": prec, "o": o, "v": v, "naux": int(v * rng.uniform(3.6, 4.4)) + 20}
        if kind == "pt":
            ntri = o * (o + 1) * (o + 2) // 6 - o
            count = min(ntri, _log_int(rng, 16, 400))
            case.update(count=count, stride=max(1, ntri // count))
        if work(case)["flops"] <= most:
            return case
        v = int(0.9 * v)


# ------------------------------------------------------------------ inputs


def _system(o, v, naux, seed):
    """eps (N,) and the symmetric factor B (naux, N, N) on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(1000003 * seed + 7919 * o + 31 * v + naux)
    N = o + v
    eo = torch.rand(o, generator=g, device=DEV, dtype=torch.float64).mul(1.2).sub(1.5).sort().values
    ev = torch.rand(v, generator=g, device=DEV, dtype=torch.float64).mul(2.9).add(0.1).sort().values
    sigma = 0.5 / math.sqrt(v * math.sqrt(naux))
    x = torch.randn(naux, N, N, generator=g, device=DEV, dtype=torch.float64).mul_(sigma)
    B = torch.triu(x)
    B += torch.triu(x, 1).transpose(1, 2)
    return torch.cat([eo, ev]), B, g


def _tri(n):
    """Row and column (row >= column) of Dalton's packed order, row-major."""
    r, c = torch.tril_indices(n, n, device=DEV)
    return r, c


def _pack(M):
    r, c = _tri(M.shape[0])
    return M[r, c]


def _unpack(p, n):
    r, c = _tri(n)
    M = torch.empty(n, n, dtype=p.dtype, device=DEV)
    M = M.index_put((r, c), p)
    return M.index_put((c, r), p)


def _amplitudes(eps, B, o, g):
    """t1 small and random, t2 of MP2, as an iteration meets them."""
    N = eps.numel()
    v, n = N - o, o * (N - o)
    Bov = B[:, :o, o:].reshape(-1, n)
    D = (eps[:o, None] - eps[None, o:]).reshape(-1)
    T = (Bov.T @ Bov) / (D[:, None] + D[None, :])
    t1 = torch.randn(n, generator=g, device=DEV, dtype=torch.float64).mul_(0.02)
    return t1, _pack(T)


def _shapes(case):
    return [tuple(int(x) for x in s.split("x")) for s in case["shapes"].split()]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ao":
        return dict(zip(("nbas", "cmo", "eri"), _ao_inputs(case, seed)), kind=kind)
    if kind == "batch":
        systems = []
        for k, (o, v) in enumerate(_shapes(case)):
            eps, B, _ = _system(o, v, 4 * v, 64 * seed + k)
            systems.append((eps.cpu().numpy(), B.cpu().numpy(), o))
        return {"kind": kind, "batch": d.CCBatch(systems), "prec": PRECISION[case["prec"]]}
    o = case["o"]
    eps, B, g = _system(o, case["v"], case["naux"], seed)
    s = {"kind": kind, "prec": PRECISION[case["prec"]], "ctx": d.CCContext(eps.cpu().numpy(), B.cpu().numpy(), o)}
    if kind in ("rhs", "grad", "pt"):
        t1, t2 = _amplitudes(eps, B, o, g)
        if kind == "pt":
            s["ctx"].set_amplitudes(t1.cpu().numpy(), t2.cpu().numpy())
            n = o * (o + 1) * (o + 2) // 6 - o
            s["slice"] = (0, case["count"] or n, case["stride"])
        else:
            s["t1"], s["t2"] = t1, t2
        if kind == "grad":
            s["t1"].requires_grad_(True)
            s["t2"].requires_grad_(True)
            s["l1"], s["l2"] = _cotangents(t1, t2, g)
    return s


def _cotangents(t1, t2, g):
    l1 = torch.randn(t1.numel(), generator=g, device=DEV, dtype=torch.float64)
    l2 = torch.randn(t2.numel(), generator=g, device=DEV, dtype=torch.float64)
    return l1, l2


def _ao_inputs(case, seed):
    """Packed pair supermatrix (positive semidefinite, eigenvalues falling off
    as those of AO integrals do) and orthonormal MO coefficients."""
    g = torch.Generator(device=DEV).manual_seed(1000003 * seed + 17 * case["nbas"] + case["rank"])
    n, r = case["nbas"], case["rank"]
    M = n * (n + 1) // 2
    X = torch.randn(r, M, generator=g, device=DEV, dtype=torch.float64)
    X *= torch.logspace(0, -4, r, device=DEV, dtype=torch.float64)[:, None]
    V = X.T @ X
    q = torch.linalg.qr(torch.randn(n, n, generator=g, device=DEV, dtype=torch.float64)).Q
    # column by column: cmo[p * nbas + a] = C[a, p]
    return n, q[:, : case["nmo"]].T.contiguous().cpu().numpy(), _pack(V).cpu().numpy()


AO_THR = 1e-6


# -------------------------------------------------------------------- runs


def run(s):
    kind = s["kind"]
    if kind == "rhs":
        with torch.no_grad():
            om1, om2 = ccsd_residual(s["ctx"], s["t1"], s["t2"], s["prec"])
        return {"om1": om1, "om2": om2}
    if kind == "grad":
        om1, om2 = ccsd_residual(s["ctx"], s["t1"], s["t2"], s["prec"])
        g1, g2 = torch.autograd.grad((om1, om2), (s["t1"], s["t2"]), (s["l1"], s["l2"]))
        return {"om1": om1, "om2": om2, "g1": g1, "g2": g2}
    if kind == "solve":
        r = s["ctx"].ccsd_energy(maxit=80, threnr=1e-9, thrvec=1e-7, precision=s["prec"])
        t1, t2 = s["ctx"].amplitudes()
        return {"e_mp2": r["e_mp2"], "e_ccsd": r["e_ccsd"], "niter": r["niter"], "t1": t1, "t2": t2}
    if kind == "pt":
        e4, e5, _, _ = s["ctx"].pt_partial(*s["slice"], precision=s["prec"])
        return {"e4": e4, "e5": e5}
    if kind == "ccsdt":
        r = s["ctx"].ccsd_energy(maxit=80, threnr=1e-9, thrvec=1e-7, precision=s["prec"])
        e4, e5 = s["ctx"].pt(s["prec"])
        t1, t2 = s["ctx"].amplitudes()
        return {"e_mp2": r["e_mp2"], "e_ccsd": r["e_ccsd"], "e4": e4, "e5": e5, "t1": t1, "t2": t2}
    if kind == "batch":
        r = s["batch"].energy(maxit=80, threnr=1e-9, thrvec=1e-7, precision=s["prec"])
        return {"e_mp2": r["e_mp2"], "e_ccsd": r["e_ccsd"], "niter": r["niter"],
                "t": [s["batch"].amplitudes(k) for k in range(s["batch"].n)]}
    return {"B": d.df_factor_ao(s["cmo"], s["eri"], s["nbas"], thr=AO_THR)}


# -------------------------------------------------------------------- work


def _residual_flops(o, v, naux):
    """Multiply-adds of one vector function, two flops each: particle ladder
    over symmetric pairs, its integrals, rings, hole ladder, ring integrals, singles."""
    return (4.0 * (v * (v + 1) // 2) ** 2 * (o * (o + 1) // 2) + naux * v**3 * (v + 1.0) + 8.0 * o**3 * v**3
            + 4.0 * o**4 * v**2 + 4.0 * naux * o**2 * v**2 + 2.0 * naux * o * v**3 + 4.0 * o**2 * v**3)


def _triples_flops(o, v, n):
    return n * (12.0 * v**4 + 12.0 * o * v**3)


def work(case):
    kind = case["kind"]
    if kind == "ao":
        M, K = case["nbas"] * (case["nbas"] + 1) // 2, case["rank"]
        n, m = case["nbas"], case["nmo"]
        return {"bytes": 8.0 * (M * (M + 1) // 2 + n * m + K * m * m),
                "flops": 1.0 * K * K * M + 2.0 * K * (n * n * m + n * m * m)}
    its = 16.0  # iterations to convergence of these systems
    if kind == "batch":
        tot = {"bytes": 0.0, "flops": 0.0}
        for o, v in _shapes(case):
            n = o * v * (o * v + 1) // 2
            tot["bytes"] += 8.0 * (4 * v * (o + v) * (o + v + 1) // 2 + n)
            tot["flops"] += its * _residual_flops(o, v, 4 * v)
        return tot
    o, v, naux = case["o"], case["v"], case["naux"]
    n, factor = o * v * (o * v + 1) // 2 + o * v, naux * (o + v) * (o + v + 1) // 2
    F, ntri = _residual_flops(o, v, naux), o * (o + 1) * (o + 2) // 6 - o
    if kind == "rhs":
        return {"bytes": 8.0 * (factor + 2 * n), "flops": F}
    if kind == "grad":
        return {"bytes": 8.0 * (factor + 4 * n), "flops": 3.0 * F}
    if kind == "solve":
        return {"bytes": 8.0 * (factor + n), "flops": its * F}
    if kind == "ccsdt":
        return {"bytes": 8.0 * (factor + n), "flops": its * F + _triples_flops(o, v, ntri)}
    return {"bytes": 8.0 * (factor + n), "flops": _triples_flops(o, v, case["count"] or ntri)}


# ------------------------------------------- the same values, plain float64


class _Plain:
    """Closed-shell CCSD in T1-dressed density-fitted form, einsum by einsum;
    amplitudes t1[i,a], t2[i,a,j,b]."""

    def __init__(self, eps, B, o):
        self.eps, self.B, self.o, self.v = eps, B, o, eps.numel() - o
        J = 2.0 * torch.einsum("Pkk->P", B[:, :o, :o])
        G = torch.einsum("Ppq,P->pq", B, J) - torch.einsum("Ppk,Pkq->pq", B[:, :, :o], B[:, :o, :])
        self.h = torch.diag(eps) - G
        self.Bov = B[:, :o, o:].contiguous()
        self.g = torch.einsum("Pkc,Pld->kcld", self.Bov, self.Bov)
        self.L = 2.0 * self.g - self.g.permute(0, 3, 2, 1)
        self.D1 = eps[:o, None] - eps[None, o:]

    def residual(self, t1, t):
        o, v, B, Bov, g = self.o, self.v, self.B, self.Bov, self.g
        N = o + v
        X, Y = torch.eye(N, dtype=B.dtype, device=DEV), torch.eye(N, dtype=B.dtype, device=DEV)
        X[:o, o:] = -t1
        Y[o:, :o] = t1.T
        Bt = torch.einsum("rp,Prs->Pps", X, B)
        Bt = torch.einsum("Pps,sq->Ppq", Bt, Y)
        F = X.T @ self.h @ Y + torch.einsum("Ppq,P->pq", Bt, 2.0 * torch.einsum("Pkk->P", Bt[:, :o, :o]))
        F = F - torch.einsum("Ppk,Pkq->pq", Bt[:, :, :o], Bt[:, :o, :])
        Bvv, Boo, Bvo = Bt[:, o:, o:].contiguous(), Bt[:, :o, :o].contiguous(), Bt[:, o:, :o].contiguous()
        u = 2.0 * t - t.permute(2, 1, 0, 3)
        om1 = torch.einsum("Pad,Pid->ia", Bvv, torch.einsum("Pkc,kcid->Pid", Bov, u))
        om1 = om1 - torch.einsum("kalc,kilc->ia", u, torch.einsum("Pki,Plc->kilc", Boo, Bov))
        om1 = om1 + torch.einsum("iakc,kc->ia", u, F[:o, o:]) + F[o:, :o].T
        om2 = torch.einsum("Pai,Pbj->iajb", Bvo, Bvo)
        tt = t.permute(1, 3, 0, 2).reshape(v * v, o * o)
        lad = []
        for a in range(v):
            Va = torch.einsum("Pc,Pbd->bcd", Bvv[:, a], Bvv).reshape(v, v * v)
            lad.append((Va @ tt).reshape(v, o, o))
        om2 = om2 + torch.stack(lad).permute(2, 0, 3, 1)
        Gam = torch.einsum("Pki,Plj->kilj", Boo, Boo) + torch.einsum("icjd,kcld->kilj", t, g)
        om2 = om2 + torch.einsum("kalb,kilj->iajb", t, Gam)
        C = torch.einsum("Pki,Pac->iakc", Boo, Bvv)
        Dm = 2.0 * torch.einsum("Pai,Pkc->iakc", Bvo, Bov) - C + 0.5 * torch.einsum("iald,ldkc->iakc", u, self.L)
        C = C - 0.5 * torch.einsum("laid,kdlc->iakc", t, g)
        X2 = -0.5 * torch.einsum("kbjc,iakc->iajb", t, C) - torch.einsum("kbic,jakc->iajb", t, C)
        X2 = X2 + 0.5 * torch.einsum("jbkc,iakc->iajb", u, Dm)
        E1 = F[o:, o:] - torch.einsum("kbld,ldkc->bc", u, g)
        E2 = F[:o, :o] + torch.einsum("lcjd,kdlc->kj", u, g)
        X2 = X2 + torch.einsum("iajc,bc->iajb", t, E1) - torch.einsum("iakb,kj->iajb", t, E2)
        return om1, om2 + X2 + X2.permute(2, 3, 0, 1)

    def energy(self, t1, t):
        return float((self.L * (t + t1[:, :, None, None] * t1[None, None])).sum())

    def solve(self):
        D2 = self.D1[:, :, None, None] + self.D1[None, None]
        t1, t = torch.zeros_like(self.D1), self.g / D2
        e_mp2 = self.energy(t1, t)
        vecs, errs = [], []
        for _ in range(80):
            om1, om2 = self.residual(t1, t)
            e = torch.cat([(om1 / self.D1).reshape(-1), (om2 / D2).reshape(-1)])
            x = torch.cat([t1.reshape(-1), t.reshape(-1)]) + e
            vecs, errs = (vecs + [x])[-8:], (errs + [e])[-8:]
            n = len(vecs)
            A = torch.full((n + 1, n + 1), -1.0, dtype=torch.float64)
            A[n, n] = 0.0
            for i in range(n):
                for j in range(i + 1):
                    A[i, j] = A[j, i] = float(errs[i] @ errs[j])
            scale = float(A[:n, :n].diagonal().max())
            if scale < 1e-26:
                break
            A[:n, :n] /= scale
            b = torch.zeros(n + 1, dtype=torch.float64)
            b[n] = -1.0
            c = torch.linalg.lstsq(A, b[:, None], driver="gelsd").solution[:n, 0]
            x = sum(float(ci) * xi for ci, xi in zip(c, vecs))
            t1, t = x[: t1.numel()].reshape(t1.shape), x[t1.numel():].reshape(t.shape)
        return e_mp2, t1, t

    def triples(self, t1, t, first, count, stride):
        """(E4, E5) of the triples i >= j >= k (i = j = k left out) of a slice of the list."""
        o, v, B = self.o, self.v, self.B
        Bvv = B[:, o:, o:].contiguous()
        q = torch.einsum("Pkc,Plj->kclj", self.Bov, B[:, :o, :o])
        ev = self.eps[o:]
        Dv = ev[:, None, None] + ev[None, :, None] + ev[None, None, :]
        Bf = Bvv.reshape(-1, v * v)
        gk = [(Bf.T @ self.Bov[:, k]).reshape(v, v, v) for k in range(o)]  # [b,d,c] = (bd|ck)

        def term(i, j, k):
            x = torch.einsum("ad,bdc->abc", t[i, :, j], gk[k])
            return x - torch.einsum("alb,cl->abc", t[i], q[k, :, :, j])

        def sym(x):
            y = 4.0 * x + x.permute(1, 2, 0) + x.permute(2, 0, 1)
            return y - 2.0 * (x.permute(0, 2, 1) + x.permute(1, 0, 2) + x.permute(2, 1, 0))

        lst = [(i, j, k) for i in range(o) for j in range(i + 1) for k in range(j + 1) if not i == j == k]
        e4 = e5 = 0.0
        for i, j, k in lst[first::stride][:count]:
            W = term(i, j, k) + term(i, k, j).permute(0, 2, 1) + term(j, i, k).permute(1, 0, 2)
            # the pair order of each term in (ai),(bj),(ck)
            W = W + term(j, k, i).permute(2, 0, 1) + term(k, i, j).permute(1, 2, 0) + term(k, j, i).permute(2, 1, 0)
            Z = t1[i][:, None, None] * self.g[j, :, k][None] + t1[j][None, :, None] * self.g[i, :, k][:, None]
            Z = Z + t1[k][None, None] * self.g[i, :, j][:, :, None]
            f = (3.0 if i == j or j == k else 6.0) / 3.0
            R = f * W / (self.eps[i] + self.eps[j] + self.eps[k] - Dv)
            e4 += (R * sym(W)).sum()
            e5 += (R * sym(Z)).sum()
        return float(e4), float(e5)


def _flat(t1, t):
    n = t1.numel()
    return t1.reshape(-1), _pack(t.reshape(n, n))


def _exact_ao(case, seed):
    n, cmo, eri = _ao_inputs(case, seed)
    M = n * (n + 1) // 2
    V = _unpack(torch.from_numpy(eri).to(DEV), M)
    dg = V.diagonal().clone()
    L = torch.zeros(M, M, dtype=torch.float64, device=DEV)
    K = 0
    while K < M:
        p = int(torch.argmax(dg))
        dp = float(dg[p])
        if dp < AO_THR:
            break
        L[K] = (V[p] - L[:K, p] @ L[:K]) / math.sqrt(dp)
        dg -= L[K] ** 2
        dg[p] = 0.0
        K += 1
    r, c = _tri(n)
    S = torch.zeros(K, n, n, dtype=torch.float64, device=DEV)
    S[:, r, c] = L[:K]
    S[:, c, r] = L[:K]
    C = torch.from_numpy(cmo).to(DEV).reshape(case["nmo"], n)
    return {"B": torch.einsum("pa,Kab,qb->Kpq", C, S, C)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "ao":
        return _exact_ao(case, seed)
    if kind == "batch":
        out = {"e_mp2": [], "e_ccsd": [], "niter": None, "t": []}
        for k, (o, v) in enumerate(_shapes(case)):
            eps, B, _ = _system(o, v, 4 * v, 64 * seed + k)
            p = _Plain(eps, B, o)
            e_mp2, t1, t = p.solve()
            out["e_mp2"].append(e_mp2)
            out["e_ccsd"].append(p.energy(t1, t))
            out["t"].append(_flat(t1, t))
        out["e_mp2"], out["e_ccsd"] = np.array(out["e_mp2"]), np.array(out["e_ccsd"])
        return out
    o, v = case["o"], case["v"]
    eps, B, g = _system(o, v, case["naux"], seed)
    p = _Plain(eps, B, o)
    if kind in ("solve", "ccsdt"):
        e_mp2, t1, t = p.solve()
        out = {"e_mp2": e_mp2, "e_ccsd": p.energy(t1, t)}
        if kind == "ccsdt":
            out["e4"], out["e5"] = p.triples(t1, t, 0, o**3, 1)
        else:
            out["niter"] = None
        out["t1"], out["t2"] = _flat(t1, t)
        return out
    t1, t2 = _amplitudes(eps, B, o, g)
    n = o * v
    if kind == "pt":
        e4, e5 = p.triples(t1.reshape(o, v), _unpack(t2, n).reshape(o, v, o, v), 0, case["count"] or o**3,
                           case["stride"])
        return {"e4": e4, "e5": e5}
    if kind == "rhs":
        om1, om2 = _flat(*p.residual(t1.reshape(o, v), _unpack(t2, n).reshape(o, v, o, v)))
        return {"om1": om1, "om2": om2}
    l1, l2 = _cotangents(t1, t2, g)
    t1.requires_grad_(True)
    t2.requires_grad_(True)
    om1, om2 = _flat(*p.residual(t1.reshape(o, v), _unpack(t2, n).reshape(o, v, o, v)))
    g1, g2 = torch.autograd.grad((om1, om2), (t1, t2), (l1, l2))
    return {"om1": om1.detach(), "om2": om2.detach(), "g1": g1, "g2": g2}
