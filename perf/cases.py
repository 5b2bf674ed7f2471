"""The work that a user of the Fock-build engine has it do, through its public entry points.

A case is a molecule family and size, a basis set, and one operation:

  jk        J[P] and K[P] from a density on the device to matrices on the device: the step of a device-resident
            SCF (FockEngine.jk_device); with "cutoff" in mixed precision, with "graph" replayed from a hipGraph,
            with "count" over a batch of molecules in one context
  g         G = J - K/2 from host memory to host memory: the drop-in for a host program's two-electron Fock call
  uhf       J[Pa + Pb], K[Pa], K[Pb], device to device: one open-shell SCF step
  gradient  the two-electron gradient per shell centre, host to host: one step of a geometry optimisation
  scf       a whole RHF from the core guess: energy and density

Geometries are those of a relaxed chain or cluster shaken by 0.01 Angstrom (a frame of an optimisation or a
dynamics run), and densities are symmetric with bond-like decay between the functions' centres; both come from the
seed alone.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "planck-refactored_amd"))

from pkfock.engine import FockEngine, PREC_MIXED  # noqa: E402
from pkfock.host import Molecule  # noqa: E402
from pkfock.molecules import alkane, water, water_cluster  # noqa: E402

ETHYLENE = ([6, 6, 1, 1, 1, 1],
            [[-0.6695, 0.0, 0.0], [0.6695, 0.0, 0.0], [-1.2321, 0.9289, 0.0], [-1.2321, -0.9289, 0.0],
             [1.2321, 0.9289, 0.0], [1.2321, -0.9289, 0.0]])


def listed():
    return [
        # the smallest call: one water in a minimal basis, every step of a long optimisation or dynamics run
        dict(name="water-sto3g", op="jk", mol="water", n=1, basis="sto-3g", engine="os", tol=1e-10),
        # one water in the double-zeta basis of the reference's examples
        dict(name="water-631gs", op="jk", mol="water", n=1, basis="6-31g*", engine="os", tol=1e-10),
        # the drop-in call of a host SCF program on a small organic molecule (50 functions)
        dict(name="ethylene-ccpvdz-host", op="g", mol="ethylene", n=1, basis="cc-pvdz", engine="os", tol=1e-10),
        # an ordinary cluster, odd size (171 functions)
        dict(name="water9-631gs", op="jk", mol="water", n=9, basis="6-31g*", engine="os", tol=1e-10),
        # a whole SCF of a small cluster: setup, one-electron integrals, some fifteen builds, diagonalisations
        dict(name="water3-631gs-scf", op="scf", mol="water", n=3, basis="6-31g*", engine="os", tol=1e-10),
        # many small molecules in one context (a conformer or training-set scan), replayed from a graph
        dict(name="water-batch-graph", op="jk", mol="water", n=6, basis="6-31g*", engine="os", tol=1e-12, count=48,
             graph=True),
        # the Rys engine forced, on an ordinary chain (185 functions)
        dict(name="c7h16-ccpvdz-rys", op="jk", mol="alkane", n=7, basis="cc-pvdz", engine="rys", tol=1e-10),
        # one geometry-optimisation step of a small chain: the gradient's integrals
        dict(name="c3h8-ccpvdz-gradient", op="gradient", mol="alkane", n=3, basis="cc-pvdz", engine="os", tol=1e-10),
        # an open-shell step with f shells (290 functions)
        dict(name="c4h10-ccpvtz-uhf", op="uhf", mol="alkane", n=4, basis="cc-pvtz", engine="os", tol=1e-10),
        # the large double-zeta chain (510 functions)
        dict(name="c20h42-ccpvdz", op="jk", mol="alkane", n=20, basis="cc-pvdz", engine="os", tol=1e-12),
        # the large triple-zeta chain with f shells (680 functions)
        dict(name="c10h22-ccpvtz", op="jk", mol="alkane", n=10, basis="cc-pvtz", engine="os", tol=1e-12),
        # the same with the small quartets in FP32
        dict(name="c10h22-ccpvtz-mixed", op="jk", mol="alkane", n=10, basis="cc-pvtz", engine="os", tol=1e-12,
             cutoff=1e-5),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: operations, families, basis sets, thresholds and sizes of the ranges above."""
    op = rng.choice(["jk", "jk", "jk", "g", "uhf", "gradient", "scf", "batch", "mixed"])
    mol = rng.choice(["water", "alkane"])
    tol = rng.choice([1e-9, 1e-10, 1e-11, 1e-12])
    engine = rng.choice(["os", "os", "auto", "rys"])
    # largest size by basis set: (water molecules, carbon atoms)
    most = {"sto-3g": (32, 30), "3-21g": (24, 24), "6-31g*": (16, 20), "cc-pvdz": (8, 16), "cc-pvtz": (3, 8)}
    basis = rng.choice(["sto-3g", "3-21g", "6-31g*", "cc-pvdz", "cc-pvdz", "cc-pvtz"])
    top = most[basis][mol == "alkane"]
    if op == "batch":
        basis = rng.choice(["sto-3g", "6-31g*", "cc-pvdz"])
        return dict(op="jk", mol="water", n=rng.randint(1, 5), basis=basis, engine=engine, tol=tol,
                    count=_log_int(rng, 2, 40), graph=rng.random() < 0.5)
    if op == "mixed":
        return dict(op="jk", mol=mol, n=_log_int(rng, 1, top), basis=basis, engine=engine, tol=tol,
                    cutoff=rng.choice([1e-4, 1e-5, 1e-6, 1e-7]))
    if op == "uhf":
        top = max(1, top // 2)
    if op == "gradient":
        top = {"sto-3g": (10, 8), "3-21g": (6, 5), "6-31g*": (4, 4), "cc-pvdz": (3, 3), "cc-pvtz": (1, 1)}[basis][mol == "alkane"]
    if op == "scf":
        basis, top = rng.choice([("sto-3g", 5), ("6-31g*", 4), ("cc-pvdz", 2)])
        mol = "water"
    case = dict(op=op, mol=mol, n=_log_int(rng, 1, top), basis=basis, engine=engine, tol=tol)
    if op == "jk" and rng.random() < 0.25:
        case["graph"] = True
    return case


# ---------------------------------------------------------------- inputs
def _geometry(case, seed, index=0):
    """Atoms and coordinates (Angstrom) of one molecule of the case."""
    rng = np.random.Generator(np.random.PCG64([int(seed) & 0x7fffffff, index]))
    if case["mol"] == "ethylene":
        Z, X = ETHYLENE
    elif case["mol"] == "alkane":
        Z, X = alkane(case["n"])
    elif case["n"] == 1 and "count" not in case:
        Z, X = water()
    elif "count" in case:  # a batch: clusters of 1..n molecules
        Z, X = water_cluster(1000 * case["n"] + index, n=1 + index % case["n"])
    else:
        Z, X = water_cluster(case["n"], n=case["n"])
    X = np.asarray(X, dtype=np.float64)
    return Z, X + rng.normal(size=X.shape) * 0.01


def _molecules(case, seed):
    return [Molecule(*_geometry(case, seed, i), case["basis"]) for i in range(case.get("count", 1))]


def _density(shells, seed, index):
    """Symmetric, one-electron occupations on the diagonal, bond-like decay (1.6 Bohr) between centres."""
    nc = [(l + 1) * (l + 2) // 2 for l in shells.l]
    x = np.repeat(shells.center, nc, axis=0)
    r = np.sqrt(((x[:, None, :] - x[None, :, :]) ** 2).sum(-1))
    rng = np.random.Generator(np.random.PCG64([int(seed) & 0x7fffffff, 7000 + index]))
    A = rng.normal(size=r.shape) * 0.25
    P = (A + A.T) * np.exp(-r / 1.6)
    P[np.diag_indices_from(P)] = rng.uniform(0.1, 1.6, size=len(r))
    return P


def prepare(case, seed):
    torch.cuda.init()
    mols = _molecules(case, seed)
    if case["op"] == "scf":
        return dict(case=case, mol=mols[0])
    shells = [m.shells() for m in mols]
    eng = FockEngine(shells if "count" in case else shells[0], case["engine"], case["tol"])
    if "cutoff" in case:
        eng.set(case["engine"], case["tol"], precision=PREC_MIXED, fp32_cutoff=case["cutoff"])
    state = dict(case=case, eng=eng)
    nd = 2 if case["op"] == "uhf" else 1
    dens = [[_density(s, seed, 100 * d + i) for i, s in enumerate(shells)] for d in range(nd)]
    if case["op"] in ("g", "gradient"):
        state["P"] = np.ascontiguousarray(dens[0][0])
        return state
    dev = torch.device("cuda:0")
    state["P"] = [torch.tensor(eng.pack(p), device=dev) for p in dens]
    state["out"] = [torch.empty_like(state["P"][0]) for _ in range(2 if nd == 1 else 3)]
    eng.set_stream(torch.cuda.current_stream(dev).cuda_stream)
    if case.get("graph"):
        eng.set_graph(True)
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "scf":
        r = state["mol"].rhf(engine=case["engine"], tol_eri=case["tol"], tol_energy=1e-11, tol_density=1e-11)
        return {"energy": r["energy"], "P": r["P"]}
    eng = state["eng"]
    if op == "g":
        return eng.g(state["P"])
    if op == "gradient":
        return eng.eri_gradient(state["P"])
    ptr = [t.data_ptr() for t in state["P"] + state["out"]]
    (eng.jk_uhf_device if op == "uhf" else eng.jk_device)(*ptr)
    return state["out"]


# ---------------------------------------------------------------- what a pass cannot do without
def _pairs(shells):
    """Every unique shell pair: class (larger l first), an estimate of its Schwarz bound from the s-type diagonal
    integral of its largest primitive pairs, and its number of primitive pairs of any weight."""
    off = np.concatenate([[0], np.cumsum(shells.nprim)])
    out = {}
    for a in range(len(shells.l)):
        for b in range(a + 1):
            ea, eb = shells.exponent[off[a]:off[a + 1], None], shells.exponent[None, off[b]:off[b + 1]]
            ca = (shells.coef * shells.prim_norm)[off[a]:off[a + 1], None]
            cb = (shells.coef * shells.prim_norm)[None, off[b]:off[b + 1]]
            z = ea + eb
            r2 = ((shells.center[a] - shells.center[b]) ** 2).sum()
            k = np.abs(ca * cb) * np.exp(-ea * eb / z * r2) * math.pi ** 1.25 * 2 ** 0.5 / z
            k = k * z ** -0.25 * (0.5 / z) ** (0.5 * (shells.l[a] + shells.l[b]))
            key = tuple(sorted((int(shells.l[a]), int(shells.l[b])), reverse=True))
            out.setdefault(key, []).append((float(k.sum()), int((k > 1e-12).sum())))
    return {key: np.array(v) for key, v in out.items()}


_work = {}


def work(case):
    """bytes: the densities in and the matrices out, once each.  flops: for every shell quartet that an estimated
    Schwarz test keeps, with K primitive quartets, n = L/2 + 1 Rys roots and Nc components,
    K [n (12 (la+lb+1)(lc+ld+1) + 3 Nc) + 20 n] + 12 Nc: 2-D recurrences, assembly, roots, and the two Coulomb and
    four exchange sums; the open-shell step has four more exchange sums, the gradient three more products of three
    factors for each of three centres.  A whole SCF counts fifteen builds."""
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _work:
        nbytes = flops = 0.0
        nmat = {"jk": 3, "g": 2, "uhf": 5, "gradient": 1, "scf": 1}[case["op"]]
        for m in _molecules(case, 0):
            s = m.shells()
            nbytes += nmat * 8.0 * s.nbasis ** 2
            cls = _pairs(s)
            for (la, lb), v in cls.items():
                for (lc, ld), w in cls.items():
                    if (la, lb) < (lc, ld):
                        continue
                    w = w[np.argsort(w[:, 0])]
                    pos = np.searchsorted(w[:, 0], case["tol"] / np.maximum(v[:, 0], 1e-300))
                    tail = np.concatenate([np.cumsum(w[::-1, 1])[::-1], [0.0]])
                    half = 0.5 if (la, lb) == (lc, ld) else 1.0
                    prim, quart = half * (v[:, 1] * tail[pos]).sum(), half * (len(w) - pos).sum()
                    n = (la + lb + lc + ld) // 2 + 1
                    nc = math.prod((l + 1) * (l + 2) // 2 for l in (la, lb, lc, ld))
                    per, dig = n * (12 * (la + lb + 1) * (lc + ld + 1) + 3 * nc + 20), 12 * nc
                    if case["op"] == "uhf":
                        dig += 8 * nc
                    if case["op"] == "gradient":
                        per += n * 27 * nc
                    flops += prim * per + quart * dig
        _work[key] = {"bytes": float(nbytes), "flops": float(flops) * (15 if case["op"] == "scf" else 1)}
    return _work[key]


# ---------------------------------------------------------------- the same in plain torch
# McMurchie-Davidson in FP64: Hermite expansions E of each primitive pair, Hermite Coulomb integrals R over the Boys
# function, the whole nb^4 tensor (or, for the gradient, its contraction differentiated by autograd).
EXACT_MAX = 60  # functions


def exact(case, seed):
    if "count" in case:
        return None
    mol = _molecules(case, seed)[0]
    s = mol.shells()
    if s.nbasis > EXACT_MAX:
        return None
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    eri = _eri(s, dev)
    n = s.nbasis
    q = torch.sqrt(torch.einsum("ijij->ij", eri).abs())
    keep = (q[:, :, None, None] * q[None, None, :, :]) >= case["tol"]
    eri = torch.where(keep, eri, torch.zeros((), dtype=eri.dtype, device=dev))
    flat, swap = eri.reshape(n * n, n * n), eri.permute(0, 2, 1, 3).reshape(n * n, n * n).contiguous()

    def jk(P):
        return (flat @ P.reshape(-1)).reshape(n, n), (swap @ P.reshape(-1)).reshape(n, n)

    if case["op"] == "scf":
        return _scf(mol, s, jk, dev)
    P = torch.tensor(_density(s, seed, 0), device=dev)
    if case["op"] == "gradient":
        G = 2 * P[:, :, None, None] * P[None, None] - P[:, None, :, None] * P[None, :, None, :]
        return _gradient(s, torch.where(keep, G, torch.zeros_like(G)), dev).cpu().numpy()
    J, K = jk(P)
    if case["op"] == "g":
        return (J - 0.5 * K).cpu().numpy()
    if case["op"] == "uhf":
        Pb = torch.tensor(_density(s, seed, 100), device=dev)
        Jb, Kb = jk(Pb)
        return [(J + Jb).reshape(-1), K.reshape(-1), Kb.reshape(-1)]
    return [J.reshape(-1), K.reshape(-1)]


def _cart(l):
    return [(x, l - x - z, z) for x in range(l, -1, -1) for z in range(l - x + 1)]


def _herm(L):
    return [(t, u, v) for t in range(L + 1) for u in range(L + 1 - t) for v in range(L + 1 - t - u)]


def _norm(c):
    df = lambda k: math.prod(range(k, 0, -2))  # noqa: E731
    return 1.0 / math.sqrt(math.prod(df(2 * k - 1) for k in c))


class _Boys(torch.autograd.Function):
    """F_0..F_M(T) along the last axis: ascending series below 36, the asymptotic form above."""

    @staticmethod
    def forward(ctx, T, M):
        F = _boys(T, M + 1)
        ctx.save_for_backward(F)
        return F[..., :M + 1].clone()

    @staticmethod
    def backward(ctx, g):
        (F,) = ctx.saved_tensors
        return -(g * F[..., 1:]).sum(-1), None


def _boys(T, M):
    Ts = T.clamp(max=36.0)
    term = torch.full_like(Ts, 1.0 / (2 * M + 1))
    s = term.clone()
    for i in range(1, 130):
        term = term * (2.0 * Ts / (2 * M + 2 * i + 1))
        s = s + term
    e = torch.exp(-Ts)
    F = [None] * (M + 1)
    F[M] = e * s
    for m in range(M, 0, -1):
        F[m - 1] = (2.0 * Ts * F[m] + e) / (2 * m - 1)
    Tl = T.clamp(min=36.0)
    g, el = 0.5 * torch.sqrt(math.pi / Tl), torch.exp(-Tl)
    big = [g]
    for m in range(M):
        g = ((2 * m + 1) * g - el) / (2 * Tl)
        big.append(g)
    return torch.stack([torch.where(T < 36.0, a, b) for a, b in zip(F, big)], -1)


def _hermite(i, j, x, a, b):
    """E_t^{i'j'} of the product of two 1-D Gaussians without its exponential, for i' <= i, j' <= j."""
    p = a + b
    pa, pb = -b * x / p, a * x / p
    E = {(0, 0): [torch.ones_like(p)]}

    def up(e, d):
        n = len(e)
        return [(e[t - 1] / (2 * p) if t >= 1 else 0) + (d * e[t] if t < n else 0) + ((t + 1) * e[t + 1] if t + 1 < n else 0)
                for t in range(n + 1)]

    for k in range(i + 1):
        if k:
            E[k, 0] = up(E[k - 1, 0], pa)
        for m in range(1, j + 1):
            E[k, m] = up(E[k, m - 1], pb)
    return E


def _prims(s, dev, centers):
    """Primitive pairs by class: exponents, centre, expansion matrix, and the contracted pair each belongs to."""
    off = np.concatenate([[0], np.cumsum(s.nprim)])
    f0 = np.concatenate([[0], np.cumsum([(l + 1) * (l + 2) // 2 for l in s.l])])
    cn = s.coef * s.prim_norm
    cls = {}
    for a in range(len(s.l)):
        for b in range(a + 1):
            A, B = (a, b) if s.l[a] >= s.l[b] else (b, a)
            cls.setdefault((int(s.l[A]), int(s.l[B])), []).append((A, B))
    out = []
    for (la, lb), lst in sorted(cls.items()):
        rows = [(k, A, B, i, j) for k, (A, B) in enumerate(lst) for i in range(off[A], off[A + 1]) for j in range(off[B], off[B + 1])]
        k, A, B, i, j = (np.array(v) for v in zip(*rows))
        t = lambda v: torch.tensor(v, dtype=torch.float64, device=dev)  # noqa: E731
        al, be, cc = t(s.exponent[i]), t(s.exponent[j]), t(cn[i] * cn[j])
        RA, RB = centers[torch.tensor(A, device=dev)], centers[torch.tensor(B, device=dev)]
        p = al + be
        P = (al[:, None] * RA + be[:, None] * RB) / p[:, None]
        x = RA - RB
        cc = cc * torch.exp(-al * be / p * (x * x).sum(1))
        E = [_hermite(la, lb, x[:, q], al, be) for q in range(3)]
        h = _herm(la + lb)
        zero = torch.zeros_like(p)
        cols = []
        for ca in _cart(la):
            for cb in _cart(lb):
                e = [E[q][ca[q], cb[q]] for q in range(3)]
                w = cc * (_norm(ca) * _norm(cb))
                cols.append(torch.stack([w * e[0][u[0]] * e[1][u[1]] * e[2][u[2]]
                                         if all(u[q] < len(e[q]) for q in range(3)) else zero for u in h], -1))
        fi = np.array([[f0[SA] + x for x in range(len(_cart(la))) for _ in _cart(lb)] for SA, _ in lst])
        fj = np.array([[f0[SB] + y for _ in _cart(la) for y in range(len(_cart(lb)))] for _, SB in lst])
        out.append(dict(l=la + lb, p=p, P=P, E=torch.stack(cols, 1), of=torch.tensor(k, device=dev), n=len(lst), h=h,
                        fi=torch.tensor(fi, device=dev), fj=torch.tensor(fj, device=dev)))
    return out


def _coulomb(b, k, i0, i1):
    """Hermite Coulomb integrals [rows i0..i1 of b][k][herm b][herm k] of two primitive-pair classes."""
    L = b["l"] + k["l"]
    p, q = b["p"][i0:i1, None], k["p"][None]
    al = p * q / (p + q)
    X = b["P"][i0:i1, None] - k["P"][None]
    F = _Boys.apply(al * (X * X).sum(-1), L)
    pre = 2.0 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q))
    lev = [{(0, 0, 0): pre * (-2.0 * al) ** m * F[..., m]} for m in range(L + 1)]
    for n in range(1, L + 1):
        for m in range(L - n + 1):
            for h in _herm(L):
                if sum(h) != n:
                    continue
                ax = max(range(3), key=lambda c: h[c])
                d = lambda c: tuple(h[z] - (c if z == ax else 0) for z in range(3))  # noqa: E731
                v = X[..., ax] * lev[m + 1][d(1)]
                if h[ax] >= 2:
                    v = v + (h[ax] - 1) * lev[m + 1][d(2)]
                lev[m][h] = v
    R = lev[0]
    rows = []
    for u in b["h"]:
        rows.append(torch.stack([R[tuple(x + y for x, y in zip(u, w))] * (-1.0) ** sum(w) for w in k["h"]], -1))
    return torch.stack(rows, -2)


def _blocks(cls, budget):
    for x, b in enumerate(cls):
        for k in cls[:x + 1]:
            size = len(k["p"]) * len(b["h"]) * max(len(k["h"]) * 3, (b["l"] + k["l"] + 1) * 60)
            step = max(1, int(budget // size))
            for i0 in range(0, len(b["p"]), step):
                yield b, k, i0, min(i0 + step, len(b["p"]))


def _eri(s, dev):
    n = s.nbasis
    out = torch.zeros(n, n, n, n, dtype=torch.float64, device=dev)
    with torch.no_grad():
        cls = _prims(s, dev, torch.tensor(s.center, device=dev))
        acc = {}
        for b, k, i0, i1 in _blocks(cls, 3e8):
            M = _coulomb(b, k, i0, i1)
            nb, nk, hb, hk = M.shape
            Y = torch.matmul(b["E"][i0:i1], M.permute(0, 2, 1, 3).reshape(nb, hb, nk * hk)).reshape(nb, -1, nk, hk)
            Y = torch.zeros(b["n"], *Y.shape[1:], dtype=Y.dtype, device=dev).index_add_(0, b["of"][i0:i1], Y)
            Z = torch.matmul(Y.permute(2, 0, 1, 3).reshape(nk, -1, hk), k["E"].transpose(1, 2).contiguous())
            Z = torch.zeros(k["n"], *Z.shape[1:], dtype=Z.dtype, device=dev).index_add_(0, k["of"], Z)
            key = (id(b), id(k))
            acc[key] = (b, k, Z + acc[key][2] if key in acc else Z)
        for b, k, Z in acc.values():
            v = Z.reshape(k["n"], b["n"], -1, k["E"].shape[1]).permute(1, 2, 0, 3)
            i, j = b["fi"][:, :, None, None], b["fj"][:, :, None, None]
            c, d = k["fi"][None, None], k["fj"][None, None]
            for x, y in ((i, j), (j, i)):
                for z, w in ((c, d), (d, c)):
                    out[x, y, z, w] = v
                    out[z, w, x, y] = v
    return out


def _gradient(s, G, dev):
    """d/d(shell centres) of 1/4 sum G (ij|kl) by autograd; G is the unsymmetrised two-particle density."""
    G = 0.125 * (G + G.transpose(0, 1))
    G = 0.5 * (G + G.transpose(2, 3))
    X = torch.tensor(s.center, device=dev, requires_grad=True)
    todo = [(x, y) for x, c in enumerate(_prims(s, dev, X.detach())) for y in range(x + 1)]
    total = torch.zeros_like(X)
    for x, y in todo:
        nb = None
        i0 = 0
        while nb is None or i0 < nb:
            cls = _prims(s, dev, X)
            b, k = cls[x], cls[y]
            nb = len(b["p"])
            step = max(1, int(4e7 // (len(k["p"]) * len(b["h"]) * max(len(k["h"]) * 3, (b["l"] + k["l"] + 1) * 60))))
            i1 = min(nb, i0 + step)
            M = _coulomb(b, k, i0, i1)
            V = torch.matmul(b["E"][i0:i1, None], M)
            V = torch.matmul(V, k["E"].transpose(1, 2)[None])
            bi, bj = b["fi"][b["of"][i0:i1]], b["fj"][b["of"][i0:i1]]
            kc, kd = k["fi"][k["of"]], k["fj"][k["of"]]
            g = G[bi[:, None, :, None], bj[:, None, :, None], kc[None, :, None], kd[None, :, None]]
            # ordered pairs that this block stands for: (ab), (ba) when the shells differ, and (cd|ab) as well
            wb = torch.where(bi[:, 0] == bj[:, 0], 1.0, 2.0).to(G.dtype)
            wk = torch.where(kc[:, 0] == kd[:, 0], 1.0, 2.0).to(G.dtype)
            w = wb[:, None] * wk[None] * (1.0 if x == y else 2.0)
            (total_x,) = torch.autograd.grad((V * g * w[:, :, None, None]).sum(), X)
            total += total_x
            i0 = i1
    return total


def _one_electron(mol, s, dev):
    """Overlap and core Hamiltonian."""
    n = s.nbasis
    cen = torch.tensor(s.center, device=dev)
    S, H = (torch.zeros(n, n, dtype=torch.float64, device=dev) for _ in range(2))
    # nuclei: Hermite Coulomb integrals against point charges
    for c in _prims(s, dev, cen):
        L = c["l"]
        p, P = c["p"], c["P"]
        V = 0
        for Zc, R in zip(mol.Z, mol.xyz):
            X = P - torch.tensor(R, device=dev)
            F = _boys(p * (X * X).sum(-1), L)
            lev = [{(0, 0, 0): (-2.0 * p) ** m * F[..., m]} for m in range(L + 1)]
            for k in range(1, L + 1):
                for m in range(L - k + 1):
                    for h in _herm(L):
                        if sum(h) == k:
                            ax = max(range(3), key=lambda z: h[z])
                            d = lambda q: tuple(h[z] - (q if z == ax else 0) for z in range(3))  # noqa: E731
                            v = X[:, ax] * lev[m + 1][d(1)]
                            lev[m][h] = v + (h[ax] - 1) * lev[m + 1][d(2)] if h[ax] >= 2 else v
            R0 = torch.stack([lev[0][h] for h in c["h"]], -1)
            V = V - float(Zc) * (2.0 * math.pi / p)[:, None] * (c["E"] * R0[:, None]).sum(-1)
        ov = c["E"][:, :, c["h"].index((0, 0, 0))] * ((math.pi / p) ** 1.5)[:, None]
        for src, dst in ((ov, S), (V, H)):
            v = torch.zeros(c["n"], src.shape[1], dtype=src.dtype, device=dev).index_add_(0, c["of"], src)
            dst[c["fi"], c["fj"]] = v
            dst[c["fj"], c["fi"]] = v
    H += _kinetic(s, cen, dev)
    return S, H


def _kinetic(s, cen, dev):
    off = np.concatenate([[0], np.cumsum(s.nprim)])
    f0 = np.concatenate([[0], np.cumsum([(l + 1) * (l + 2) // 2 for l in s.l])])
    cn = s.coef * s.prim_norm
    T = np.zeros((s.nbasis, s.nbasis))
    for A in range(len(s.l)):
        for B in range(len(s.l)):
            la, lb = int(s.l[A]), int(s.l[B])
            al = torch.tensor(s.exponent[off[A]:off[A + 1], None] + 0 * s.exponent[None, off[B]:off[B + 1]])
            be = torch.tensor(s.exponent[None, off[B]:off[B + 1]] + 0 * al.numpy())
            w = torch.tensor(cn[off[A]:off[A + 1], None] * cn[None, off[B]:off[B + 1]])
            x = torch.tensor(s.center[A] - s.center[B])
            p = al + be
            E = [_hermite(la, lb + 2, x[q] + 0 * p, al, be) for q in range(3)]
            w = w * torch.exp(-al * be / p * (x * x).sum()) * (math.pi / p) ** 1.5
            for i, a in enumerate(_cart(la)):
                for j, b in enumerate(_cart(lb)):
                    o = lambda q, d: E[q][a[q], b[q] + d][0] if b[q] + d >= 0 else torch.zeros_like(p)  # noqa: E731
                    t = 0
                    for q in range(3):
                        k = -2.0 * be * be * o(q, 2) + be * (2 * b[q] + 1) * o(q, 0) - 0.5 * b[q] * (b[q] - 1) * o(q, -2)
                        for z in range(3):
                            if z != q:
                                k = k * o(z, 0)
                        t = t + k
                    T[f0[A] + i, f0[B] + j] = float((w * t).sum()) * _norm(a) * _norm(b)
    return torch.tensor(T, device=dev)


def _scf(mol, s, jk, dev):
    """RHF with DIIS from the core guess, to an error of 1e-12."""
    S, H = _one_electron(mol, s, dev)
    nocc = int(sum(mol.Z)) // 2
    e, U = torch.linalg.eigh(S)
    X = U * e.rsqrt() @ U.T

    def occupied(F):
        _, C = torch.linalg.eigh(X @ F @ X)
        C = (X @ C)[:, :nocc]
        return 2.0 * C @ C.T

    P, Fs, errs = occupied(H), [], []
    for _ in range(200):
        J, K = jk(P)
        F = H + J - 0.5 * K
        energy = 0.5 * float(((H + F) * P).sum())
        err = X @ (F @ P @ S - S @ P @ F) @ X
        if float(err.abs().max()) < 1e-12:
            break
        Fs, errs = (Fs + [F])[-8:], (errs + [err])[-8:]
        m = len(Fs)
        B = -torch.ones(m + 1, m + 1, dtype=torch.float64)
        B[m, m] = 0.0
        for i in range(m):
            for j in range(m):
                B[i, j] = float((errs[i] * errs[j]).sum())
        B[:m, :m] /= B[:m, :m].abs().max()
        rhs = torch.zeros(m + 1, dtype=torch.float64)
        rhs[m] = -1.0
        c = torch.linalg.lstsq(B, rhs[:, None], driver="gelsd").solution[:, 0]
        P = occupied(sum(float(c[i]) * Fs[i] for i in range(m)))
    rep = sum(float(mol.Z[i] * mol.Z[j]) / float(np.linalg.norm(mol.xyz[i] - mol.xyz[j]))
              for i in range(len(mol.Z)) for j in range(i))
    return {"energy": energy + rep, "P": P.cpu().numpy()}
