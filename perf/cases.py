"""The work a user of this library has it do, as measurable cases.

A case is a dict of plain values; ``prepare`` makes what a program holds before
the call, ``run`` is one pass through the public entry points, ``work`` the
bytes and operations the pass cannot do without, and ``exact`` the same results
from plain torch and numpy in 64 bits (McMurchie-Davidson integrals over the
embedded basis data, a textbook RHF on top of them), where that is quick.

Kinds of case:
  jk       one Fock build's J and K for a given density: through device
           pointers (a program that keeps D, J, K in HBM) or host buffers (the
           drop-in for rchem's JK_direct)
  scf      a molecule from its geometry to a converged energy and density, as a
           scan or a geometry step calls it: the basis is new on every pass
  grad     the same with the analytic nuclear gradient
  batch    many small molecules solved together
  oneel    S, T and V
  tensor   the full two-electron tensor (rchem's build_I)
"""
import ctypes
import json
import math
import os

import numpy as np
import torch

import rchem_amd
from rchem_amd import basis as rb
from rchem_amd._lib import PREC_FP64, PREC_MIXED, default_opts, lib
from rchem_amd.inputs import nocc_of, water_cluster

# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def jk(name, waters, basis, precision="fp64", path="device", shells=0):
    return {"name": name, "kind": "jk", "waters": waters, "shells": shells, "basis": basis,
            "precision": precision, "path": path}


def scf(name, waters, basis, precision="fp64", diis=8, graph=True, purify=True, kind="scf"):
    return {"name": name, "kind": kind, "waters": waters, "basis": basis, "precision": precision,
            "diis": diis, "graph": graph, "purify": purify}


def listed():
    return [
        # the smallest call: rchem's own test system (7 functions), latency and launches
        jk("jk_water1_sto3g", 1, "STO-3G"),
        # the drop-in call of a small cluster: host buffers, 104 functions
        jk("jk_water8_host", 8, "6-31G", path="host"),
        # the headline build, 832 functions, all FP64 and with FP32 for the small quartets
        jk("jk_water64", 64, "6-31G"),
        jk("jk_water64_mixed", 64, "6-31G", precision="mixed"),
        # s, p and d shells of the synthetic integral benchmark, at its density
        jk("jk_spd", 0, "", shells=210),
        # rchem's whole program: plain iterations, eigensolver, 7 functions
        scf("scf_water1_sto3g", 1, "STO-3G", diis=0, graph=False, purify=False),
        # a small cluster with the defaults a user reaches for: DIIS and an eigensolver
        scf("scf_water8", 8, "6-31G", graph=False, purify=False),
        # a larger one with every device-side option on
        scf("scf_water32_mixed", 32, "6-31G", precision="mixed"),
        # a step of a geometry optimisation
        scf("grad_water12", 12, "6-31G", graph=False, kind="grad"),
        # many small closed-shell systems of uneven size in one call
        {"name": "batch_48", "kind": "batch", "molecules": 48, "largest": 12, "precision": "fp64"},
        # one-electron matrices of the headline system
        {"name": "oneel_water64", "kind": "oneel", "waters": 64, "basis": "6-31G"},
        # the tensor of a small molecule, for a program that keeps integrals
        {"name": "tensor_water3", "kind": "tensor", "waters": 3, "basis": "6-31G"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["jk", "jk", "jk", "spd", "scf", "grad", "batch", "oneel", "tensor"])
    basis = rng.choice(["STO-3G", "6-31G", "6-31G"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "jk":
        c = jk("", _log_int(rng, 1, 64), basis, precision, rng.choice(["device", "host"]))
    elif kind == "spd":
        c = jk("", 0, "", precision, rng.choice(["device", "host"]), shells=_log_int(rng, 8, 200))
    elif kind == "scf":
        diis = rng.choice([6, 8])
        c = scf("", _log_int(rng, 1, 28), basis, precision, diis, rng.random() < 0.5,
                rng.random() < 0.5)
    elif kind == "grad":
        c = scf("", _log_int(rng, 1, 12), basis, "fp64", 8, False, rng.random() < 0.5, kind="grad")
    elif kind == "batch":
        c = {"kind": "batch", "molecules": rng.randint(5, 48), "largest": rng.randint(2, 12),
             "precision": precision}
    elif kind == "oneel":
        c = {"kind": "oneel", "waters": _log_int(rng, 1, 64), "basis": basis}
    else:
        c = {"kind": "tensor", "waters": _log_int(rng, 1, 4), "basis": basis}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _cluster(waters, seed):
    """(H2O)_waters on the benchmark's jittered lattice, filled cell by cell."""
    side = max(1, math.ceil(round(waters ** (1 / 3), 9)))
    Z, xyz = water_cluster(dims=(side, side, side), seed=seed)
    return Z[:3 * waters], np.ascontiguousarray(xyz[:3 * waters])


def _synthetic(shells, seed):
    """The integral benchmark's shells at its density (2000 in a 20-bohr cube), its shares of
    s, p and d (0.5, 0.35, 0.15) taken exactly, so that every seed has the same functions."""
    rng = np.random.default_rng(seed)
    box = 20.0 * (shells / 2000.0) ** (1 / 3)
    centres = rng.uniform(0.0, box, (shells, 3))
    np_, nd = int(0.35 * shells + 0.5), int(0.15 * shells + 0.5)
    ls = rng.permutation(np.repeat([0, 1, 2], [shells - np_ - nd, np_, nd])).astype(np.int32)
    exps = np.exp(rng.uniform(math.log(0.1), math.log(100.0), (shells, 3)))
    coefs = rng.uniform(0.1, 1.0, (shells, 3))
    for a, c, l in zip(exps, coefs, ls):  # unit self-overlap of the x^l component
        c /= math.sqrt(c @ (2.0 * np.sqrt(np.outer(a, a)) / np.add.outer(a, a)) ** (l + 1.5) @ c)
    return centres, ls, np.full(shells, 3, dtype=np.int32), exps.reshape(-1), coefs.reshape(-1)


def _molecules(case, seed):
    """Clusters of 1 .. largest waters, every size about equally often."""
    rng = np.random.default_rng(seed)
    sizes = rng.permutation(np.arange(case["molecules"]) % case["largest"] + 1)
    return [_cluster(int(w), int(rng.integers(1 << 31))) for w in sizes]


def _shells(Z, xyz, basis):
    """Shells (centre, l, exponents, coefficients) in the library's order."""
    path = os.path.join(os.path.dirname(rchem_amd.__file__), "data", basis.lower() + ".json")
    with open(path) as fh:
        elements = json.load(fh)["elements"]
    out = []
    for z, r in zip(Z, np.asarray(xyz).reshape(-1, 3)):
        for s in elements[str(z)]["electron_shells"]:
            ex = [float(e) for e in s["exponents"]]
            rows = s["coefficients"]
            for k, l in enumerate(s["angular_momentum"]):
                out.append((r, l, ex, [float(c) for c in rows[min(k, len(rows) - 1)]]))
    return out


def _case_shells(case, seed):
    if case.get("shells"):
        xyz, ls, npr, ex, cf = _synthetic(case["shells"], seed)
        ends = np.cumsum(npr)
        return [(xyz[s], int(ls[s]), list(ex[ends[s] - npr[s]:ends[s]]),
                 list(cf[ends[s] - npr[s]:ends[s]])) for s in range(len(ls))]
    Z, xyz = _cluster(case["waters"], seed)
    return _shells(Z, xyz, case["basis"])


def _ncart(l):
    return (l + 1) * (l + 2) // 2


def _density(shells, seed):
    """A symmetric density with the falloff of a closed-shell molecule's: entries of order one
    on an atom, decaying exponentially with the distance of the two functions' centres."""
    rng = np.random.default_rng([seed, 1])
    at = np.concatenate([np.tile(r, (_ncart(l), 1)) for r, l, _, _ in shells])
    n = len(at)
    far = np.sqrt(((at[:, None] - at[None]) ** 2).sum(-1))
    D = rng.standard_normal((n, n)) * 0.3
    D = (D + D.T) * np.exp(-0.7 * far)
    D[np.arange(n), np.arange(n)] = rng.uniform(0.2, 1.0, n)
    return D


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------


def _opts(case):
    return default_opts(precision=PREC_MIXED if case.get("precision") == "mixed" else PREC_FP64)


def _basis(case, seed, ctx):
    if case.get("shells"):
        return rb.Basis.from_shells(*_synthetic(case["shells"], seed), ctx=ctx)
    Z, xyz = _cluster(case["waters"], seed)
    return rb.Basis.new(Z, xyz, case["basis"], ctx=ctx)


def prepare(case, seed):
    torch.zeros(1, device="cuda")  # torch loads the HIP runtime, the library shares it
    ctx = rb.Context(0)
    s = {"case": case, "ctx": ctx}
    kind = case["kind"]
    if kind == "jk":
        s["basis"] = _basis(case, seed, ctx)
        D = _density(_case_shells(case, seed), seed)
        s["opts"] = _opts(case)
        if case["path"] == "device":
            s["D"] = torch.from_numpy(D).cuda()
            s["J"], s["K"] = torch.zeros_like(s["D"]), torch.zeros_like(s["D"])
        else:
            s["D"], s["J"], s["K"] = D, np.zeros_like(D), np.zeros_like(D)
    elif kind in ("scf", "grad"):
        s["Z"], s["xyz"] = _cluster(case["waters"], seed)
        s["opts"] = _opts(case)
    elif kind == "batch":
        s["molecules"] = _molecules(case, seed)
        s["opts"] = _opts(case)
    else:
        s["Z"], s["xyz"] = _cluster(case["waters"], seed)
        s["basis"] = _basis(case, seed, ctx)
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "jk":
        if case["path"] == "host":
            rb.JK_direct(s["J"], s["K"], s["basis"], s["D"], s["opts"])
        else:
            ptr = [ctypes.c_void_p(s[k].data_ptr()) for k in "DJK"]
            ctx.check(lib().rchem_jk_device(ctx.h, *ptr, ctypes.byref(s["opts"])))
        # the two-electron part of the Fock matrix, what every caller forms next
        return {"J": s["J"], "K": s["K"], "G": 2.0 * s["J"] - s["K"]}
    if kind in ("scf", "grad"):
        B = rb.Basis.new(s["Z"], s["xyz"], case["basis"], ctx=ctx)
        kw = dict(nocc=nocc_of(s["Z"]), opts=s["opts"], diis=case["diis"], graph=case["graph"],
                  purify=case["purify"])
        if kind == "scf":
            res, D = rb.scf(B, s["xyz"], s["Z"], **kw)
            return {"e": np.array([res.e_elec, res.e_total]), "D": D}
        res, g = rb.rhf_gradient(B, s["xyz"], s["Z"], **kw)
        return {"e": np.array([res.e_elec, res.e_total]), "grad": g}
    if kind == "batch":
        res = rb.batch_scf(s["molecules"], "STO-3G", thresh_e=1e-10, max_iter=128, diis=8,
                           opts=s["opts"], ctx=ctx, graph=True)
        return {"e_elec": np.array([r.e_elec for r in res]),
                "e_total": np.array([r.e_total for r in res]),
                "converged": np.array([r.converged for r in res])}
    if kind == "oneel":
        S, T, V = rb.one_electron(s["basis"], s["xyz"], s["Z"])
        return {"S": S, "T": T, "V": V}
    return {"I": rb.build_I(s["basis"])}


# ---------------------------------------------------------------------------
# the work of a pass
# ---------------------------------------------------------------------------

_EVERY = [(la, lb) for la in range(3) for lb in range(la + 1)]


def _pairs(shells):
    """Per shell pair (a >= b): class, significant primitive pairs, and a bound of the size of
    sqrt((ab|ab)) from s functions of the same exponents."""
    n = len(shells)
    at = np.array([s[0] for s in shells])
    own = [i for i, s in enumerate(shells) for _ in s[2]]
    al = np.array([a for s in shells for a in s[2]])
    co = np.array([abs(c) * (2 * a / math.pi) ** 0.75 for s in shells for a, c in zip(s[2], s[3])])
    own = np.array(own)
    cnt, q = np.zeros((n, n)), np.zeros((n, n))
    for lo in range(0, len(al), 256):
        o = slice(lo, lo + 256)
        far = ((at[own[o]][:, None] - at[own][None]) ** 2).sum(-1)
        z = al[o][:, None] + al[None]
        k = co[o][:, None] * co[None] * 5.914967172795613 / z * np.exp(
            -al[o][:, None] * al[None] / z * far)
        idx = (np.broadcast_to(own[o][:, None], k.shape), np.broadcast_to(own[None], k.shape))
        np.add.at(cnt, idx, k > 1e-15)
        np.add.at(q, idx, k / (2 * z) ** 0.25)
    a, b = np.tril_indices(n)
    l = np.array([s[1] for s in shells])
    hi, lo = np.maximum(l[a], l[b]), np.minimum(l[a], l[b])
    return hi * (hi + 1) // 2 + lo, cnt[a, b], q[a, b]


def _build_flops(shells, tau=1e-12):
    """Operations of one Fock build: every unique quartet whose bound reaches tau."""
    cls, npp, q = _pairs(shells)
    total = 0.0
    for X, (la, lb) in enumerate(_EVERY):
        for Y, (lc, ld) in enumerate(_EVERY[:X + 1]):
            bra, ket = cls == X, cls == Y
            if not bra.any() or not ket.any():
                continue
            order = np.argsort(-q[ket])
            qs = q[ket][order]
            ps = np.concatenate([[0.0], np.cumsum(npp[ket][order])])
            m = np.searchsorted(-qs, -tau / np.maximum(q[bra], 1e-300))
            half = 0.5 if X == Y else 1.0
            quartets, prims = half * m.sum(), half * (npp[bra] * ps[m]).sum()
            e = sum(_ncart(l) for l in range(la, la + lb + 1))
            f = sum(_ncart(l) for l in range(lc, lc + ld + 1))
            comp = _ncart(la) * _ncart(lb) * _ncart(lc) * _ncart(ld)
            # a primitive quartet: its prefactors and Boys functions, three operations for each
            # [e0|f0]; a contracted one: six J/K updates for each integral
            total += prims * (50 + 3 * e * f) + quartets * 12 * comp
    return float(total)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        flops = nbytes = 0.0
        for Z, xyz in _molecules(case, 1):
            sh = _shells(Z, xyz, "STO-3G")
            n = sum(_ncart(s[1]) for s in sh)
            flops += 10 * _build_flops(sh) + 10 * 20 * n ** 3  # ten iterations at the least
            nbytes += 8 * (4 * len(Z) + 3)
        return {"bytes": nbytes, "flops": flops}
    sh = _case_shells(case, 1)
    n = sum(_ncart(s[1]) for s in sh)
    data = 8 * sum(5 + 2 * len(s[2]) for s in sh)
    if kind == "jk":
        return {"bytes": data + 24 * n * n, "flops": _build_flops(sh)}
    if kind == "scf":
        return {"bytes": data + 8 * n * n, "flops": 10 * (_build_flops(sh) + 20 * n ** 3)}
    if kind == "grad":  # the derivative integrals: nine blocks, about three builds
        return {"bytes": data + 8 * len(sh), "flops": 10 * (1.3 * _build_flops(sh) + 20 * n ** 3)}
    cls, npp, _ = _pairs(sh)
    if kind == "oneel":  # a primitive pair and nucleus: a Boys function and its Hermite sum
        comp = np.array([_ncart(a) * _ncart(b) for a, b in _EVERY])
        return {"bytes": data + 24 * n * n,
                "flops": float((npp * 3 * case["waters"] * (40 + 6 * comp[cls])).sum())}
    return {"bytes": data + 8 * n ** 4, "flops": float(_build_flops(sh, 1e-40))}


# ---------------------------------------------------------------------------
# the same results in 64 bits, without this library
# ---------------------------------------------------------------------------

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_F = dict(dtype=torch.float64, device=_DEV)


def _boys_values(m_max, T):
    """F_0 .. F_m_max: the all-positive series and downward recursion below 36, the asymptote
    and upward recursion above."""
    small = T < 36.0
    t = torch.where(small, T, torch.zeros_like(T))
    e = torch.exp(-t)
    term = torch.full_like(t, 1.0 / (2 * m_max + 1))
    total = term.clone()
    top = float(t.max()) if t.numel() else 0.0
    for k in range(1, 400):
        term = term * (2 * t / (2 * m_max + 2 * k + 1))
        total += term
        if k % 8 == 0 and 2 * top < 2 * m_max + 2 * k + 1 and float(term.max()) < 1e-18:
            break
    lo = [None] * (m_max + 1)
    lo[m_max] = e * total
    for m in range(m_max - 1, -1, -1):
        lo[m] = (2 * t * lo[m + 1] + e) / (2 * m + 1)
    u = torch.where(small, torch.full_like(T, 36.0), T)
    eu = torch.exp(-u)
    hi = [torch.sqrt(math.pi / u) / 2 * torch.erf(torch.sqrt(u))]
    for m in range(m_max):
        hi.append(((2 * m + 1) * hi[m] - eu) / (2 * u))
    return [torch.where(small, a, b) for a, b in zip(lo, hi)]


class _Boys(torch.autograd.Function):
    """dF_m/dT = -F_(m+1)."""

    @staticmethod
    def forward(ctx, m_max, T):
        F = _boys_values(m_max + 1, T)
        ctx.save_for_backward(*F[1:])
        return tuple(F[:-1])

    @staticmethod
    def backward(ctx, *g):
        return None, -sum(x * f for x, f in zip(g, ctx.saved_tensors))


def _boys(m_max, T):
    return _Boys.apply(m_max, T) if T.requires_grad else _boys_values(m_max, T)


def _hermite_coulomb(L, alpha, X):
    """R_tuv(alpha, X), t + u + v <= L, as a dict of tensors."""
    F = _boys(L, alpha * (X[0] * X[0] + X[1] * X[1] + X[2] * X[2]))
    cur = {}
    for n in range(L, -1, -1):
        new = {(0, 0, 0): (-2 * alpha) ** n * F[n]}
        for total in range(1, L - n + 1):
            for t in range(total + 1):
                for u in range(total - t + 1):
                    k = [t, u, total - t - u]
                    i = next(x for x in range(3) if k[x] > 0)
                    k1 = list(k)
                    k1[i] -= 1
                    v = X[i] * cur[tuple(k1)]
                    if k1[i] > 0:
                        k2 = list(k1)
                        k2[i] -= 1
                        v = v + k1[i] * cur[tuple(k2)]
                    new[tuple(k)] = v
        cur = new
    return cur


def _hermite_e(la, lb, a, b, ab):
    """E_t^ij of one axis, i <= la, j <= lb, without the Gaussian prefactor of the pair."""
    p = a + b
    pa, pb = -b / p * ab, a / p * ab
    E = {(0, 0, 0): torch.ones_like(p)}

    def get(i, j, t):
        return E.get((i, j, t), torch.zeros_like(p))

    for i in range(la + 1):
        for j in range(lb + 1):
            if i == j == 0:
                continue
            for t in range(i + j + 1):
                if i > 0:
                    v = get(i - 1, j, t - 1) / (2 * p) + pa * get(i - 1, j, t) + \
                        (t + 1) * get(i - 1, j, t + 1)
                else:
                    v = get(i, j - 1, t - 1) / (2 * p) + pb * get(i, j - 1, t) + \
                        (t + 1) * get(i, j - 1, t + 1)
                E[(i, j, t)] = v
    return E


def _components(l):
    """xx, xy, xz, yy, yz, zz: the library's order."""
    return [(i, j, l - i - j) for i in range(l, -1, -1) for j in range(l - i, -1, -1)]


def _tuv(L):
    return [(t, u, k - t - u) for k in range(L + 1) for t in range(k, -1, -1)
            for u in range(k - t, -1, -1)]


def _fact2(n):
    return 1 if n <= 1 else n * _fact2(n - 2)


def _norm(l, a):
    return math.sqrt(2.0 ** (2 * l + 1.5) * a ** (l + 1.5) / math.pi ** 1.5)


def _comp_norm(c):
    return 1.0 / math.sqrt(math.prod(_fact2(2 * i - 1) for i in c))


class _Pairs:
    """The primitive pairs of all shell pairs of one class (la >= lb) with their Hermite
    expansions E[prim, component pair, tuv]; `row` is each primitive's shell pair, `at` the
    shells' centres."""

    def __init__(self, shells, at, f0, la, lb):
        self.la, self.lb = la, lb
        self.shells = [(i, j) for i, s in enumerate(shells) for j, r in enumerate(shells)
                       if s[1] == la and r[1] == lb and (la != lb or i >= j)]
        if not self.shells:
            return
        prim = [(i, j, x, y, cx * cy * _norm(la, x) * _norm(lb, y), k)
                for k, (i, j) in enumerate(self.shells)
                for x, cx in zip(*shells[i][2:]) for y, cy in zip(*shells[j][2:])]
        i, j, al, be, co, row = (np.array(v) for v in zip(*prim))
        c = np.array([s[0] for s in shells])
        keep = np.abs(co) * np.exp(-al * be / (al + be) * ((c[i] - c[j]) ** 2).sum(1)) > 1e-25
        i, j, row = (torch.tensor(v[keep], device=_DEV) for v in (i, j, row))
        al, be, co = (torch.tensor(v[keep], **_F) for v in (al, be, co))
        A, B = at[i], at[j]
        self.row, self.al, self.be, self.p = row, al, be, al + be
        self.AB = A - B
        self.pre = co * torch.exp(-al * be / self.p * (self.AB * self.AB).sum(1))
        self.P = (al[:, None] * A + be[:, None] * B) / self.p[:, None]
        self.ca, self.cb = _components(la), _components(lb)
        self.tuv = _tuv(la + lb)
        ax = [_hermite_e(la, lb, al, be, self.AB[:, x]) for x in range(3)]
        zero = torch.zeros_like(self.p)
        self.E = torch.stack([torch.stack([
            self.pre * (_comp_norm(ca) * _comp_norm(cb)) * ax[0].get((ca[0], cb[0], t), zero) *
            ax[1].get((ca[1], cb[1], u), zero) * ax[2].get((ca[2], cb[2], v), zero)
            for t, u, v in self.tuv], 1) for ca in self.ca for cb in self.cb], 1)
        # the basis functions of every (shell pair, component pair)
        self.fa = np.array([[f0[x] + u for u in range(len(self.ca)) for _ in self.cb]
                            for x, _ in self.shells])
        self.fb = np.array([[f0[y] + v for _ in self.ca for v in range(len(self.cb))]
                            for _, y in self.shells])

    def functions(self):
        return [torch.tensor(v.reshape(-1), device=_DEV) for v in (self.fa, self.fb)]


def _layout(shells, at=None):
    """The pair classes and the number of functions."""
    f0, n = [], 0
    for s in shells:
        f0.append(n)
        n += _ncart(s[1])
    if at is None:
        at = torch.tensor(np.array([s[0] for s in shells]), **_F)
    lmax = max(s[1] for s in shells)
    cls = [_Pairs(shells, at, f0, la, lb) for la in range(lmax + 1) for lb in range(la + 1)]
    return [c for c in cls if c.shells], n


def _one_electron_class(c, C, Z):
    """S, T and V of one pair class: [shell pair, component pair] each."""
    p = c.p
    ax = [_hermite_e(c.la, c.lb + 2, c.al, c.be, c.AB[:, x]) for x in range(3)]
    zero = torch.zeros_like(p)

    def s1(x, i, j):
        return ax[x].get((i, j, 0), zero) if j >= 0 else zero

    def t1(x, i, j):
        return (-2 * c.be ** 2 * s1(x, i, j + 2) + c.be * (2 * j + 1) * s1(x, i, j) -
                0.5 * j * (j - 1) * s1(x, i, j - 2))

    pre = c.pre * (math.pi / p) ** 1.5
    s, t = [], []
    for ca in c.ca:
        for cb in c.cb:
            nrm = _comp_norm(ca) * _comp_norm(cb) * pre
            o = [s1(x, ca[x], cb[x]) for x in range(3)]
            k = [t1(x, ca[x], cb[x]) for x in range(3)]
            s.append(nrm * o[0] * o[1] * o[2])
            t.append(nrm * (k[0] * o[1] * o[2] + o[0] * k[1] * o[2] + o[0] * o[1] * k[2]))
    v = []
    step = max(1, (1 << 22) // len(C))
    for lo in range(0, len(p), step):
        o = slice(lo, lo + step)
        X = [c.P[o, x][:, None] - C[None, :, x] for x in range(3)]
        R = _hermite_coulomb(c.la + c.lb, p[o][:, None].expand_as(X[0]), X)
        h = torch.stack([(R[k] * Z).sum(1) for k in c.tuv], 1)
        v.append(-2 * math.pi / p[o][:, None] * (c.E[o] * h[:, None, :]).sum(2))
    shape = (len(c.shells), len(s))
    return [torch.zeros(shape, **_F).index_add(0, c.row, x)
            for x in (torch.stack(s, 1), torch.stack(t, 1), torch.cat(v))]


def _one_electron(shells, Z, xyz):
    cls, n = _layout(shells)
    Zt = torch.tensor(np.asarray(Z, dtype=float), **_F)
    C = torch.tensor(np.asarray(xyz, dtype=float).reshape(-1, 3), **_F)
    out = [np.zeros((n, n)) for _ in range(3)]
    for c in cls:
        for M, v in zip(out, _one_electron_class(c, C, Zt)):
            M[c.fa, c.fb] = M[c.fb, c.fa] = v.cpu().numpy()
    return out


def _eri_blocks(b, k, rows):
    """(ab|cd) of bra primitives `rows` with every ket primitive, kets contracted:
    [bra primitive, bra components, ket shell pair, ket components]."""
    nb, nk = b.E.shape[1], k.E.shape[1]
    p, q = b.p[rows][:, None], k.p[None]
    X = [b.P[rows, i][:, None] - k.P[None, :, i] for i in range(3)]
    R = _hermite_coulomb(b.la + b.lb + k.la + k.lb, (p * q / (p + q)).expand_as(X[0]), X)
    pre = 2 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q))
    h = 0.0
    for j, tk in enumerate(k.tuv):
        g = torch.stack([R[(t[0] + tk[0], t[1] + tk[1], t[2] + tk[2])] * pre for t in b.tuv], 1)
        y = torch.matmul(b.E[rows], g)  # bra primitive, bra components, ket primitive
        h = h + y[..., None] * ((-1.0) ** sum(tk) * k.E[None, None, :, :, j])
    return torch.zeros((len(p), nb, len(k.shells), nk), **_F).index_add(2, k.row, h)


def _bra_steps(b, k, most=1 << 24):
    step = max(1, most // (len(k.p) * b.E.shape[1] * k.E.shape[1] +
                           len(k.p) * len(_tuv(b.la + b.lb + k.la + k.lb))))
    return [slice(lo, lo + step) for lo in range(0, len(b.p), step)]


def _eri(shells):
    """The full tensor (ab|cd)."""
    cls, n = _layout(shells)
    I = torch.zeros((n, n, n, n), **_F)
    for x, b in enumerate(cls):
        for k in cls[:x + 1]:
            M = torch.zeros((len(b.shells), b.E.shape[1], len(k.shells), k.E.shape[1]), **_F)
            for o in _bra_steps(b, k, 1 << 26):
                M.index_add_(0, b.row[o], _eri_blocks(b, k, o))
            ab = [v[:, None] for v in b.functions()]
            cd = [v[None] for v in k.functions()]
            M = M.reshape(len(ab[0]), -1)
            for p, q in (ab, ab[::-1]):
                for r, s in (cd, cd[::-1]):
                    I[p, q, r, s] = M
                    I[r, s, p, q] = M
    return I


def _gradient(shells, atom, Z, xyz, D, W):
    """dE/dR by differentiating the integrals contracted with D and W."""
    R = torch.tensor(np.asarray(xyz, dtype=float).reshape(-1, 3), **_F, requires_grad=True)
    Zt = torch.tensor(np.asarray(Z, dtype=float), **_F)
    D, W = torch.as_tensor(D, **_F), torch.as_tensor(W, **_F)
    cls, _ = _layout(shells, R[torch.tensor(atom, device=_DEV)])
    far = R[:, None] - R[None] + torch.eye(len(R), **_F)[..., None]
    e = 0.5 * ((Zt[:, None] * Zt[None]) * (1 - torch.eye(len(R), **_F)) /
               torch.sqrt((far * far).sum(-1))).sum()
    for c in cls:
        fa, fb = c.functions()
        twice = torch.tensor([2.0 if i != j else 1.0 for i, j in c.shells], **_F)
        S, T, V = _one_electron_class(c, R, Zt)
        d, w = (M[fa, fb].reshape(S.shape) * twice[:, None] for M in (D, W))
        e = e + (2 * d * (T + V)).sum() - (2 * w * S).sum()
    for x, b in enumerate(cls):
        for k in cls[:x + 1]:
            (a, b2), (c, d) = b.functions(), k.functions()
            G = 2 * D[a, b2][:, None] * D[c, d][None] - 0.5 * (
                D[a][:, c] * D[b2][:, d] + D[a][:, d] * D[b2][:, c])
            G = G.reshape(len(b.shells), b.E.shape[1], len(k.shells), k.E.shape[1])
            tb, tk = (torch.tensor([2.0 if i != j else 1.0 for i, j in v.shells], **_F)
                      for v in (b, k))
            G = G * tb[:, None, None, None] * tk[:, None] * (1.0 if b is k else 2.0)
            leaves = [[t.detach().requires_grad_() for t in (v.P, v.E)] for v in (b, k)]
            keep = [(v.P, v.E) for v in (b, k)]
            for v, (P, E) in zip((b, k), leaves):
                v.P, v.E = P, E
            for o in _bra_steps(b, k):
                (_eri_blocks(b, k, o) * G[b.row[o]]).sum().backward()
            for v, (P, E) in zip((b, k), keep):
                v.P, v.E = P, E
            for old, new in zip(keep, leaves if b is not k else [leaves[1]]):
                for t, l in zip(old, new):
                    if l.grad is not None:
                        e = e + (t * l.grad).sum() - (t * l.grad).sum().detach()
    e.backward()
    return R.grad.cpu().numpy()


def _jk_of(I, D):
    D = torch.as_tensor(D, **_F)
    n = len(D)
    J = (I.reshape(n * n, n * n) @ D.reshape(-1)).reshape(n, n)
    K = (I.permute(0, 2, 1, 3).reshape(n * n, n * n) @ D.reshape(-1)).reshape(n, n)
    return J.cpu().numpy(), K.cpu().numpy()


def _rhf(shells, Z, xyz):
    """Closed-shell SCF (DIIS over eight Fock matrices) to the limit of 64 bits: the electronic
    and total energies, D, and W = D F D."""
    S, T, V = _one_electron(shells, Z, xyz)
    I = _eri(shells)
    H, nocc = T + V, nocc_of(Z)
    w, U = np.linalg.eigh(S)
    X = (U / np.sqrt(w)) @ U.T
    Fs, es = [], []
    F = H
    for _ in range(80):
        C = X @ np.linalg.eigh(X.T @ F @ X)[1][:, :nocc]
        D = C @ C.T
        J, K = _jk_of(I, D)
        F0 = H + 2 * J - K
        e = float((D * (H + F0)).sum())
        err = X.T @ (F0 @ D @ S - S @ D @ F0) @ X
        if np.abs(err).max() < 1e-12:
            break
        Fs, es = (Fs + [F0])[-8:], (es + [err])[-8:]
        m = len(Fs)
        B = -np.ones((m + 1, m + 1))
        B[m, m] = 0
        B[:m, :m] = [[(x * y).sum() for y in es] for x in es]
        B[:m, :m] /= B[:m, :m].max()
        c = np.linalg.lstsq(B, np.r_[np.zeros(m), -1.0], rcond=None)[0][:m]
        F = sum(x * f for x, f in zip(c, Fs))
    R = np.asarray(xyz).reshape(-1, 3)
    nuc = sum(Z[i] * Z[j] / np.linalg.norm(R[i] - R[j]) for i in range(len(Z)) for j in range(i))
    return e, e + nuc, D, D @ F0 @ D


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return None
    shells = _case_shells(case, seed)
    n = sum(_ncart(s[1]) for s in shells)
    if kind == "oneel":
        Z, xyz = _cluster(case["waters"], seed)
        return dict(zip("STV", _one_electron(shells, Z, xyz)))
    # beyond these sizes the tensor (or its derivative's graph) takes too long
    if n > (60 if case.get("shells") or kind == "grad" else 110):
        return None
    if kind == "jk":
        J, K = _jk_of(_eri(shells), _density(shells, seed))
        return {"J": J, "K": K, "G": 2.0 * J - K}
    if kind == "tensor":
        return {"I": _eri(shells).cpu().numpy()}
    Z, xyz = _cluster(case["waters"], seed)
    e, total, D, W = _rhf(shells, Z, xyz)
    if kind == "scf":
        return {"e": np.array([e, total]), "D": D}
    where = {tuple(r): i for i, r in enumerate(xyz)}
    g = _gradient(shells, [where[tuple(s[0])] for s in shells], Z, xyz, D, W)
    return {"e": np.array([e, total]), "grad": g}
