"""Performance cases: what users of this framework have it do, from one water to
a batch of 32 forty-water clusters, through the entry points of myqc_amd.

The molecules are clusters of waters at the density of the 40-water workload
(40 waters in a 12 A cube), optionally with a few helium atoms between them, so
that the basis size n = 7 waters + helium takes ragged values too.

  solve         one RHF solve from a geometry: the system, one-electron
                integrals, screened two-electron integrals, (the learned
                density), the SCF loop and the density of its orbitals
  lockstep      many clusters of one size, set up and solved by ManySolver
  integrals     a new geometry: its screened integrals and one Fock build
  fock          one Fock build G(D) from stored integrals
  fock_uhf      the two spin Fock builds of a UHF iteration
  eri_full      the dense integrals of the int2e program, to host memory
  ao2mo         the (ia|jb) records of the ao2mo program, to host memory
  mp2           the transform kept on the device, then the MP2 energies
  batch         RHF of many small molecules in one persistent launch
  mlp_gradient  forward and backward pass of the learned guess's network
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

from myqc_amd import guess as G
from myqc_amd import molecules as M
from myqc_amd.basis import build_basis, read_ftab
from myqc_amd.hip import BF16X3, FP32, FP64, Context, enuc
from myqc_amd.many import ManySolver

TOL = 1e-12          # Schwarz threshold of every stored build
MLP_IN, MLP_WIDTH, MLP_OUT = 200, 128, 16   # the shipped network's layers


# -- the cases ---------------------------------------------------------------
def listed():
    return [
        # the smallest solve a user runs: one molecule, where launches, copies and host work are everything
        dict(name="solve_1_water", kind="solve", waters=1, helium=0, precision="fp64", learned=False),
        # an ordinary molecule of a geometry scan, every step in double precision
        dict(name="solve_8_waters", kind="solve", waters=8, helium=0, precision="fp64", learned=False),
        # a large single system the fast way: learned start and FP32 increments, ragged n
        dict(name="solve_24_waters_mixed", kind="solve", waters=24, helium=3, precision="mixed", learned=True),
        # the headline workload: 32 clusters of 40 waters set up and solved together
        dict(name="lockstep_32x40_waters", kind="lockstep", waters=40, helium=0, systems=32, precision="mixed",
             learned=True),
        # int2e followed by one RHFI2G for a new geometry, at the headline size
        dict(name="integrals_40_waters", kind="integrals", waters=40, helium=0),
        # RHFI2G alone, called by a program with its own SCF loop
        dict(name="fock_40_waters", kind="fock", waters=40, helium=0),
        # UHFI2G on an ordinary system with ragged n
        dict(name="fock_uhf_13_waters", kind="fock_uhf", waters=13, helium=4),
        # the XX record of an int2e run
        dict(name="eri_full_5_waters", kind="eri_full", waters=5, helium=0),
        # the ijab records of an ao2mo run, in the mixed-precision option
        dict(name="ao2mo_9_waters_bf16x3", kind="ao2mo", waters=9, helium=0, precision="bf16x3"),
        # the MP2 workload of the benchmark, in double precision
        dict(name="mp2_24_waters", kind="mp2", waters=24, helium=0, precision="fp64"),
        # screening: a thousand clusters of 2-5 waters, as the training data of the learned guess is made
        dict(name="batch_1024_clusters", kind="batch", molecules=1024),
        # one training step of the learned guess on a large minibatch
        dict(name="mlp_gradient_8192", kind="mlp_gradient", rows=8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "lockstep", "integrals", "fock", "fock_uhf", "eri_full", "ao2mo", "mp2",
                       "batch", "mlp_gradient"])
    helium = rng.randint(0, 6)
    if kind == "solve":
        return dict(kind=kind, waters=_log_int(rng, 1, 40), helium=helium, precision=rng.choice(["fp64", "mixed"]),
                    learned=rng.random() < 0.5)
    if kind == "lockstep":
        return dict(kind=kind, waters=_log_int(rng, 4, 40), helium=rng.randint(0, 2), systems=rng.randint(2, 32),
                    precision=rng.choice(["fp64", "mixed"]), learned=rng.random() < 0.5)
    if kind in ("integrals", "fock", "fock_uhf"):
        return dict(kind=kind, waters=_log_int(rng, 1, 40), helium=helium)
    if kind == "eri_full":
        return dict(kind=kind, waters=_log_int(rng, 1, 6), helium=helium)
    if kind == "ao2mo":
        return dict(kind=kind, waters=rng.randint(1, 9), helium=helium, precision=rng.choice(["fp64", "bf16x3"]))
    if kind == "mp2":
        return dict(kind=kind, waters=_log_int(rng, 3, 24), helium=helium, precision=rng.choice(["fp64", "bf16x3"]))
    if kind == "batch":
        return dict(kind=kind, molecules=_log_int(rng, 32, 1024))
    return dict(kind=kind, rows=_log_int(rng, 100, 16384))


# -- inputs ------------------------------------------------------------------
def _cluster(waters, helium, seed):
    """(Z, xyz in bohr): the waters, then the helium atoms, no heavy atom or
    helium nearer than 2.6 A to another."""
    box = 12.0 * ((waters + 0.5 * helium) / 40.0) ** (1.0 / 3.0)
    Z, x = M.water_cluster(waters, seed=seed, box=box)
    rng = np.random.default_rng([seed, 1])
    heavy = [x[3 * k] for k in range(waters)]
    Z, x, edge = list(Z), list(x), box
    while helium > 0:
        p = rng.uniform(0.0, edge, size=3)
        if min(np.linalg.norm(p - q) for q in heavy) >= 2.6:
            heavy.append(p)
            x.append(p)
            Z.append(2)
            helium -= 1
        else:
            edge *= 1.002   # a crowded box grows until the atom fits
    return Z, M.to_bohr(Z, np.array(x))


def _orbitals(n, block, seed):
    """n orthonormal columns, mostly within blocks of `block` functions (as
    localised orbitals are), or without structure (block 0)."""
    rng = np.random.default_rng([seed, 2])
    A = rng.normal(size=(n, n))
    if block:
        i = np.arange(n) // block
        A = np.where(i[:, None] == i[None, :], A, 0.02 * A)
    return np.linalg.qr(A)[0]


def _energies(n, nocc, seed):
    rng = np.random.default_rng([seed, 3])
    return np.concatenate([np.sort(rng.uniform(-20.0, -0.4, nocc)), np.sort(rng.uniform(0.3, 3.0, n - nocc))])


def _prec(case):
    return {"fp64": FP64, "mixed": FP32, "bf16x3": BF16X3}[case["precision"]]


def _mlp_inputs(rows, seed):
    """Rows like the pair features (one-hot elements, radial and neighbour
    Gaussians, zero padding) with targets and masks."""
    rng = np.random.default_rng([seed, 4])
    X = np.zeros((rows, MLP_IN), np.float32)
    r = np.arange(rows)
    X[r, rng.choice([0, 7], rows)] = 1.0
    X[r, 10 + rng.choice([0, 7], rows)] = 1.0
    X[:, 20:36] = np.exp(-0.5 * ((rng.uniform(0.0, 8.0, (rows, 1)) - 0.5 * np.arange(16)) / 0.5) ** 2)
    X[:, 37:197] = rng.uniform(0.0, 1.5, (rows, 160)) * (rng.random((rows, 160)) < 0.2)
    T = rng.normal(0.0, 0.3, (rows, MLP_OUT)).astype(np.float32)
    K = (rng.random((rows, MLP_OUT)) < 0.6).astype(np.float32)
    return X, T, K


def _mlp_weights(seed):
    """The flat parameter vector: per layer the weights (out x in), uniform
    within the Xavier bound, then small biases."""
    rng = np.random.default_rng([seed, 5])
    dims, p = [MLP_IN, MLP_WIDTH, MLP_WIDTH, MLP_WIDTH, MLP_OUT], []
    for a, b in zip(dims, dims[1:]):
        p += [rng.uniform(-1.0, 1.0, a * b) * math.sqrt(6.0 / (a + b)), rng.normal(0.0, 0.05, b)]
    return np.concatenate(p).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "lockstep":
        s["mols"] = [_cluster(case["waters"], case["helium"], 1000 * seed + k) for k in range(case["systems"])]
        s["solver"] = ManySolver(k=case["systems"], learned=case["learned"], precision=_prec(case))
        return s
    ctx = s["ctx"] = Context(0)
    if kind == "batch":
        # as many clusters of each size, whatever the seed, in mixed order
        per = [G.water_clusters((case["molecules"] + 5 - w) // 4, 10 * seed + w, w, w) for w in (2, 3, 4, 5)]
        ctx.batch_set([per[k % 4][k // 4] for k in range(case["molecules"])])
        return s
    if kind == "mlp_gradient":
        ctx.mlp_create(MLP_IN, MLP_WIDTH, MLP_OUT, 0)
        ctx.mlp_params(set_to=_mlp_weights(seed))
        s["XTM"] = _mlp_inputs(case["rows"], seed)
        return s
    Z, xyz = s["Z"], s["xyz"] = _cluster(case["waters"], case["helium"], seed)
    basis, ftab = s["basis"], s["ftab"] = build_basis(Z), read_ftab()
    n, nocc = basis.norb, sum(Z) // 2
    s["nocc"] = nocc
    if kind == "solve":
        if case["learned"] and not G.load(ctx):
            raise RuntimeError("no trained network in the package")
        return s
    if kind != "integrals":
        ctx.set_system(Z, xyz, basis, ftab)
    if kind in ("fock", "fock_uhf"):
        ctx.eri_build(TOL)
    if kind in ("integrals", "fock", "fock_uhf"):
        C = _orbitals(n, 7, seed)
        Ca, Cb = C[:, :nocc], C[:, :nocc - 1]
        s["D"], s["Da"], s["Db"] = 2.0 * Ca @ Ca.T, Ca @ Ca.T, Cb @ Cb.T
    if kind in ("ao2mo", "mp2"):
        s["C"], s["eig"] = _orbitals(n, 0, seed), _energies(n, nocc, seed)
    return s


# -- one pass ----------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "lockstep":
        # the orbitals' signs (and mixtures of degenerate ones) are not unique, so they stay out
        res = next(s["solver"].solve([s["mols"]], want_orbitals=True))
        return dict(E=np.array([r["E"] for r in res]), eig=np.array([r["eig"] for r in res]))
    ctx = s["ctx"]
    if kind == "solve":
        ctx.set_system(s["Z"], s["xyz"], s["basis"], s["ftab"])
        S, H = ctx.int1e()
        ctx.eri_build(TOL)
        D0 = ctx.guess_density(s["Z"], s["xyz"]) if case["learned"] else None
        r = ctx.rhf(H, S, s["nocc"], enuc(s["Z"], s["xyz"]), D_guess=D0, precision=_prec(case))
        return dict(E=r["E"], eig=r["eig"], D=ctx.density(r["C"], s["nocc"]), S=S, H=H)
    if kind == "integrals":
        ctx.set_system(s["Z"], s["xyz"], s["basis"], s["ftab"])
        stored = ctx.eri_build(TOL)
        return dict(stored=stored, G=ctx.fock_G(s["D"]))
    if kind == "fock":
        return ctx.fock_G(s["D"])
    if kind == "fock_uhf":
        return ctx.fock_G_uhf(s["Da"], s["Db"])
    if kind == "eri_full":
        return ctx.eri_full(0.0)
    if kind == "ao2mo":
        return ctx.ao2mo(s["C"], s["nocc"], _prec(case))
    if kind == "mp2":
        ctx.ao2mo(s["C"], s["nocc"], _prec(case), download=False)
        return np.array(ctx.mp2(s["eig"], s["nocc"]))
    if kind == "batch":
        E, _, conv = ctx.batch_rhf()
        return dict(E=E, converged=conv, D=np.concatenate([d.ravel() for d in ctx.batch_density()]))
    return ctx.mlp_gradient(*s["XTM"])


# -- the work a pass cannot do without ----------------------------------------
def _unique(n):
    """Unique integrals above the Schwarz threshold: every pair of functions
    of a small system, about 34 partners per function in a large one at this
    density (45.2 M integrals for 40 waters)."""
    pairs = min(0.5 * n * (n + 1), 34.0 * n)
    return 0.5 * pairs * (pairs + 1)


def work(case):
    kind = case["kind"]
    if kind == "mlp_gradient":
        w = MLP_IN * MLP_WIDTH + 2 * MLP_WIDTH ** 2 + MLP_WIDTH * MLP_OUT
        r = case["rows"]
        # forward, weight gradients, and input gradients of all layers but the first
        return dict(bytes=4.0 * (r * (MLP_IN + 2 * MLP_OUT) + 2 * w), flops=2.0 * r * (3 * w - MLP_IN * MLP_WIDTH))
    if kind == "batch":
        n = 24.5   # mean size of 2-5 waters
        per = 1000.0 * _unique(n) + 10 * (12.0 * _unique(n) + 20 * 2.0 * n ** 3)
        return dict(bytes=8.0 * case["molecules"] * 3 * n * n, flops=case["molecules"] * per)
    n, nocc = 7 * case["waters"] + case["helium"], 5 * case["waters"] + case["helium"]
    nv, u = n - nocc, _unique(n)
    # about 1000 operations per contracted integral (81 primitive quartets), 12 per integral of a Fock build
    eri = 1000.0 * u
    if kind in ("solve", "lockstep"):
        k = case.get("systems", 1)
        # ten Fock builds over the stored integrals, ten densities of twenty products
        return dict(bytes=k * 8.0 * (10 * u + 6.0 * n * n), flops=k * (eri + 120.0 * u + 10 * 25 * 2.0 * n ** 3))
    if kind == "integrals":
        return dict(bytes=8.0 * (2 * u + 2.0 * n * n), flops=eri + 12.0 * u)
    if kind == "fock":
        return dict(bytes=8.0 * (u + 2.0 * n * n), flops=12.0 * u)
    if kind == "fock_uhf":
        return dict(bytes=8.0 * (u + 4.0 * n * n), flops=20.0 * u)
    if kind == "eri_full":
        return dict(bytes=8.0 * n ** 4, flops=1000.0 * n ** 4 / 8)
    # four quarter steps from the unique integrals, the first two over pairs of the other side
    steps = 1.0 * (nocc * n ** 4 + nocc * nv * n ** 3) + 2.0 * (nocc ** 2 * nv * n ** 2 + (nocc * nv) ** 2 * n)
    out = 8.0 * (nocc * nv) ** 2
    return dict(bytes=n ** 4 + out, flops=steps + 1000.0 * n ** 4 / 8)


# -- the same in plain 64-bit arithmetic ---------------------------------------
# Contracted s and p shells by McMurchie-Davidson, with the conventions that fix
# the values: pi in single precision, the tabulated Boys function with its
# expansion orders, and primitive quartets below 1e-14 left out.
PI_SP = float(np.float32(3.1415926535897931))
STO3G_1S = [0.1543290, 0.5353281, 0.4446345]
STO3G = {1: [(0, STO3G_1S, [3.4252509, 0.6239137, 0.1688554], 0)],
         2: [(0, STO3G_1S, [6.3624214, 1.1589230, 0.3136498], 0)],
         8: [(0, STO3G_1S, [130.7093214, 23.8088661, 6.4436083], 0),
             (0, [-0.0999672, 0.3995128, 0.7001155], [5.0331513, 1.1695961, 0.3803890], 1),
             (1, [0.1559163, 0.6076837, 0.3919574], [5.0331513, 1.1695961, 0.3803890], 1)]}
HERM = [(0, 0, 0)] + [t for d in (1, 2) for t in
                      [(a, b, d - a - b) for a in range(d, -1, -1) for b in range(d - a, -1, -1)]]


def _boys(Q, T, ft, mmax):
    """F_0..F_mmax(T) at expansion order Q (a tensor like T)."""
    Tk = torch.floor(10.0 * T.clamp(max=12.0) + 0.5).clamp(max=120.0)
    x = Tk / 10.0 - T
    at = Tk.long() * 23 + Q
    f = torch.zeros_like(T)
    for k in range(6, -1, -1):
        f = f * x / (k + 1) + ft[at + k]   # Horner form of sum_k Ft(Tk, Q + k) x^k / k!
    e = torch.exp(-T)
    low = [torch.zeros_like(T) for _ in range(mmax + 1)]
    for j in range(12, -1, -1):
        f = torch.where(Q > j, (2.0 * T * f + e) / (2 * j + 1), f)
        if j <= mmax:
            low[j] = torch.where(Q >= j, f, low[j])
    iT = 1.0 / T.clamp(min=1.0)
    c = torch.tensor([[0.4999489092, -0.2473631686, 0.321180909, -0.3811559346], [0.4998436875, -0.24249438, 0.24642845, 0],
                      [0.499093162, -0.2152832, 0, 0], [0.490, 0, 0, 0]], dtype=T.dtype, device=T.device)
    c = c[(T >= 15).long() + (T >= 18).long() + (T >= 24).long()]
    g = ((c[..., 3] * iT + c[..., 2]) * iT + c[..., 1]) * iT + c[..., 0]
    es = torch.where(T < 2.0 * Q + 36.0, e, torch.zeros_like(e))
    up = [0.5 * math.sqrt(PI_SP) * iT.sqrt() - es * g * iT]
    for j in range(1, mmax + 1):
        up.append(0.5 * iT * ((2 * j - 1) * up[-1] - es))
    return [torch.where(T < 12.0, a, b) for a, b in zip(low, up)]


def _hermite_r(alpha, R, F):
    """R_tuv up to order 4 for every element, as a dict."""
    r = {(m, 0, 0, 0): (-2.0 * alpha) ** m * F[m] for m in range(5)}
    for d in range(1, 5):
        for t in range(d, -1, -1):
            for u in range(d - t, -1, -1):
                k = [t, u, d - t - u]
                ax = 0 if k[0] else 1 if k[1] else 2
                k[ax] -= 1
                l = list(k)
                l[ax] -= 1
                for m in range(5 - d):
                    v = R[ax] * r[(m + 1, *k)]
                    if k[ax]:
                        v = v + k[ax] * r[(m + 1, *l)]
                    r[(m, t, u, d - t - u)] = v
    return {k[1:]: v for k, v in r.items() if k[0] == 0}


def _dense_eri(Z, xyz, device):
    """(ij|kl) over unordered function pairs, as a matrix, and the index
    (i, j) -> pair."""
    ft = np.fromfile(os.path.join("myqc_amd", "data", "Ftab"), dtype="<f8", offset=4, count=121 * 23)
    ft = torch.tensor(ft.reshape(23, 121).T.copy().ravel(), device=device)
    shells, ao = [], 0
    for z, R in zip(Z, xyz):
        for l, cs, al, bl in STO3G[z]:
            norm = [(2 * a / PI_SP) ** 0.75 if l == 0 else (128 * a ** 5 / PI_SP ** 3) ** 0.25 for a in al]
            shells.append((l, np.array(cs) * norm, np.array(al), bl, R, ao))
            ao += 2 * l + 1
    n = ao
    p, P, eij, bl, E = [], [], [], [], []
    owner, rows = [], []
    for a, (la, ca, aa, ba, A, oa) in enumerate(shells):
        for lb, cb, ab, bb, B, ob in shells[a:]:
            for x in range(2 * la + 1):
                for y in range(2 * lb + 1):
                    if oa == ob and x > y:
                        continue
                    rows.append((oa + x, ob + y))
                    owner.append(len(p))
                    blk = np.zeros((9, 10))
                    for q, (i, j) in enumerate((i, j) for i in range(3) for j in range(3)):
                        s = aa[i] + ab[j]
                        C = (aa[i] * A + ab[j] * B) / s
                        k = math.exp(-aa[i] * ab[j] * float((A - B) @ (A - B)) / s) * ca[i] * cb[j]
                        ex = []   # Hermite coefficients along each axis
                        for d in range(3):
                            v = [1.0, 0.0, 0.0]
                            for on, X in ((la == 1 and x == d, A), (lb == 1 and y == d, B)):
                                if on:
                                    w = C[d] - X[d]
                                    v = [w * v[0] + v[1], v[0] / (2 * s) + w * v[1] + 2 * v[2], v[1] / (2 * s) + w * v[2]]
                            ex.append(v)
                        blk[q] = [k * ex[0][t] * ex[1][u] * ex[2][v] for t, u, v in HERM]
                    E.append(blk)
            s = (aa[:, None] + ab[None, :]).ravel()
            p.append(s)
            P.append(((aa[:, None, None] * A + (ab[None, :, None] * B)).reshape(9, 3)) / s[:, None])
            eij.append(np.exp(-(aa[:, None] * ab[None, :]).ravel() / s * float((A - B) @ (A - B))))
            bl.append(ba + bb)
    t = lambda v: torch.tensor(np.array(v), dtype=torch.float64, device=device)
    p, P, eij, E = t(p), t(P), t(eij), t(E)
    bl = torch.tensor(bl, device=device)
    owner = torch.tensor(owner, device=device)
    S, N = len(p), len(rows)
    pk, Pk, ek = p.reshape(1, -1), P.reshape(1, -1, 3), eij.reshape(1, -1)
    sign = t([(-1.0) ** sum(h) for h in HERM])
    Ek = (E * sign).contiguous()                       # N x 9 x 10
    out = torch.empty(N, N, dtype=torch.float64, device=device)
    for b0 in range(0, S, 32):
        b1 = min(S, b0 + 32)
        pb, Pb, eb = p[b0:b1].reshape(-1, 1), P[b0:b1].reshape(-1, 1, 3), eij[b0:b1].reshape(-1, 1)
        Q = 3 * (bl[b0:b1].repeat_interleave(9)[:, None] + bl.repeat_interleave(9)[None, :])
        alpha = pb * pk / (pb + pk)
        R = Pb - Pk
        F = _boys(Q, alpha * (R * R).sum(-1), ft, 4)
        pre = 2.0 * PI_SP ** 2.5 / (pb * pk * torch.sqrt(pb + pk)) * (eb * ek >= 1.0e-14)
        r = _hermite_r(alpha, [R[..., d] for d in range(3)], F)
        mine = torch.nonzero((owner >= b0) & (owner < b1)).ravel()
        Eb = E[mine]                                   # m x 9 x 10
        acc = torch.zeros(len(mine), N, dtype=torch.float64, device=device)
        for hb, (t0, u0, v0) in enumerate(HERM):
            if not bool((Eb[:, :, hb] != 0).any()):
                continue
            # the ket side contracted first: sum over its primitives and Hermite functions
            ket = torch.zeros((b1 - b0) * 9, N, dtype=torch.float64, device=device)
            for hk, (t1, u1, v1) in enumerate(HERM):
                V = (pre * r[(t0 + t1, u0 + u1, v0 + v1)]).reshape(-1, S, 9)
                for k in range(9):
                    ket += V[:, owner, k] * Ek[:, k, hk]
            ket = ket.reshape(b1 - b0, 9, N)
            for k in range(9):
                acc += Eb[:, k, hb, None] * ket[owner[mine] - b0, k]
        out[mine] = acc
    at = torch.zeros(n, n, dtype=torch.long, device=device)
    for m, (i, j) in enumerate(rows):
        at[i, j] = at[j, i] = m
    return out, at


def exact(case, seed):
    kind = case["kind"]
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "mlp_gradient":
        par = torch.tensor(_mlp_weights(seed), dtype=torch.float64, device=device, requires_grad=True)
        X, T, K = (torch.tensor(a, dtype=torch.float64, device=device) for a in _mlp_inputs(case["rows"], seed))
        dims, o, h = [MLP_IN, MLP_WIDTH, MLP_WIDTH, MLP_WIDTH, MLP_OUT], 0, X
        for l in range(4):
            W = par[o:o + dims[l] * dims[l + 1]].reshape(dims[l + 1], dims[l])
            o += dims[l] * dims[l + 1]
            h = h @ W.T + par[o:o + dims[l + 1]]
            o += dims[l + 1]
            h = torch.nn.functional.silu(h) if l < 3 else h
        loss = (K * (h - T) ** 2).sum() / K.sum()
        loss.backward()
        return loss.item(), par.grad
    # a whole SCF has no closed value, and larger systems take too long
    n = 7 * case.get("waters", 99) + case.get("helium", 0)
    if kind not in ("integrals", "fock", "fock_uhf", "eri_full", "ao2mo", "mp2") or n > 69:
        return None
    Z, xyz = _cluster(case["waters"], case["helium"], seed)
    pairs, at = _dense_eri(Z, xyz, device)
    nocc = sum(Z) // 2
    XX = pairs[at.reshape(-1)][:, at.reshape(-1)].reshape(n, n, n, n)   # (ij|kl)
    if kind == "eri_full":
        return XX
    t = lambda v: torch.tensor(v, dtype=torch.float64, device=device)
    if kind in ("integrals", "fock", "fock_uhf"):
        C = t(_orbitals(n, 7, seed))
        Da, Db = C[:, :nocc] @ C[:, :nocc].T, C[:, :nocc - 1] @ C[:, :nocc - 1].T
        J = lambda D: (XX.reshape(n * n, n * n) @ D.reshape(-1)).reshape(n, n)
        K = lambda D: (XX.permute(0, 2, 1, 3).reshape(n * n, n * n) @ D.reshape(-1)).reshape(n, n)
        if kind == "fock_uhf":
            return J(Da + Db) - K(Da), J(Da + Db) - K(Db)
        Gm = J(2 * Da) - K(2 * Da) / 2
        return dict(stored=None, G=Gm) if kind == "integrals" else Gm
    C, eig = t(_orbitals(n, 0, seed)), t(_energies(n, nocc, seed))
    o, v = C[:, :nocc], C[:, nocc:]
    nv = n - nocc
    half = (o.T @ XX.reshape(n, -1)).reshape(nocc, n, n * n).transpose(1, 2).contiguous() @ v   # i, kl, a
    half = half.reshape(nocc, n, n, nv).permute(0, 3, 1, 2).contiguous()                        # i, a, k, l
    iajb = (half.transpose(2, 3).contiguous() @ o).transpose(2, 3).contiguous() @ v             # i, a, j, b
    if kind == "ao2mo":
        return iajb
    den = eig[:nocc, None, None, None] - eig[None, nocc:, None, None] + eig[None, None, :nocc, None] - eig[nocc:]
    x = iajb - iajb.permute(0, 3, 2, 1)
    aa = float((x * x / den).sum()) / 4
    ab = float((iajb * iajb / den).sum())
    return torch.tensor([aa, ab, 2 * aa + ab], dtype=torch.float64)
