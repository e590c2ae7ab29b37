"""Cases of the performance measurements: the calls that a program built on
this library makes, over the sizes and options that it meets.

A case is one kind of call on one molecule (cc-pVDZ) or one batch of them:

* fock    a Fock build with a new density, G = 2J(D) - K(D): put, commit,
          compute, get (the step that every SCF iteration repeats); `nden`
          densities at once (spin or response densities), `tau` > 0 the
          mixed-precision build
* purify  the purification of a Fock matrix to a density (the other half of
          an SCF iteration)
* batch   one Fock build of many small molecules at once
* scf     the first iterations of a batched SCF: builds, DIIS, purification
* setup   what a program pays for a new geometry before its first build:
          pairs, screening and tiles, overlap, core Hamiltonian, S^-1/2
* eri     a list of shell quartets through the integral interface

The molecules are those of gtfock_amd.geometry (water and water clusters,
all-trans alkanes, hydrogen-capped graphene flakes) with bonds scaled by
`stretch`, as along a potential curve, and atoms displaced by the seed, so
that another seed is another geometry, density or Fock matrix.
"""
import itertools
import math
import os
import tempfile

import numpy as np
import torch

import gtfock_amd as g
from gtfock_amd import geometry

GBS = os.path.join(g.DATA_DIR, "cc-pvdz.gbs")
BOHR = 1.0 / 0.529177210903
CHARGE = {"H": 1, "C": 6, "N": 7, "O": 8}


def listed():
    return [
        # the smallest call: launch and copy latency, 24 functions
        dict(name="fock water", kind="fock", mol="water", size=1, stretch=1.0, nden=1, tau=0.0),
        # a small organic molecule, 114 functions
        dict(name="fock benzene", kind="fock", mol="flake", size=1, stretch=1.0, nden=1, tau=0.0),
        # a cluster with the two densities of an unrestricted build
        dict(name="fock water cluster, 2 densities", kind="fock", mol="water", size=7, stretch=1.0, nden=2, tau=0.0),
        # the headline molecule, 250 functions
        dict(name="fock C10H22", kind="fock", mol="alkane", size=10, stretch=1.0, nden=1, tau=0.0),
        # coronene in the mixed-precision option, 396 functions
        dict(name="fock C24H12 mixed", kind="fock", mol="flake", size=2, stretch=1.0, nden=1, tau=1e-4),
        # the largest single build, 846 functions
        dict(name="fock C54H18", kind="fock", mol="flake", size=3, stretch=1.0, nden=1, tau=0.0),
        # a batch of alkanes and water clusters, half each
        dict(name="batch 40 molecules", kind="batch", count=40, largest=9, stretch=1.0),
        # start of a batched SCF of small molecules
        dict(name="scf 12 molecules", kind="scf", count=12, largest=4, stretch=1.0, iters=5),
        # purification at the headline size (launch latency) and at the largest
        dict(name="purify C10H22", kind="purify", mol="alkane", size=10, stretch=1.0),
        dict(name="purify C54H18", kind="purify", mol="flake", size=3, stretch=1.0),
        # a new geometry of coronene
        dict(name="setup C24H12", kind="setup", mol="flake", size=2, stretch=1.0),
        # integrals of listed quartets for a program's own use
        dict(name="eri benzene", kind="eri", mol="flake", size=1, stretch=1.0, nquartets=30000),
    ]


def draw(rng):
    kind = rng.choice(["fock", "fock", "fock", "fock", "batch", "scf", "purify", "purify", "setup", "eri"])
    case = dict(kind=kind, stretch=round(rng.uniform(0.98, 1.06), 4))
    if kind in ("batch", "scf"):
        small = kind == "scf"
        case["count"] = int(round(math.exp(rng.uniform(math.log(3), math.log(16 if small else 48)))))
        case["largest"] = rng.randint(2, 5 if small else 9)
        if small:
            case["iters"] = rng.randint(3, 6)
        return case
    mol = rng.choice(["water", "alkane", "flake"])
    top = {"water": 12, "alkane": 16, "flake": 2}[mol]
    if kind == "purify" and mol == "flake":
        top = 3
    if kind == "eri":
        top = {"water": 6, "alkane": 5, "flake": 1}[mol]
    case["mol"] = mol
    case["size"] = min(top, int(math.exp(rng.uniform(0.0, math.log(top + 1.0)))))
    if kind == "fock":
        case["nden"] = rng.choice([1, 1, 1, 2, 3])
        case["tau"] = rng.choice([0.0, 0.0, 1e-4])
    if kind == "eri":
        case["nquartets"] = int(round(math.exp(rng.uniform(math.log(50), math.log(40000)))))
    return case


# ---- inputs ---------------------------------------------------------------------


def _atoms(mol, size, stretch, rng):
    if mol == "water":
        atoms = geometry.water() if size == 1 else geometry.water_cluster(size, rng)
    elif mol == "alkane":
        atoms = geometry.alkane(size)
    else:
        atoms = geometry.graphene_flake(size)
    move = rng.normal(scale=0.01, size=(len(atoms), 3))
    return [(s, tuple(float(v) for v in stretch * np.array(x) + m)) for (s, x), m in zip(atoms, move)]


def _basis(atoms):
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "mol.xyz")
        with open(path, "w") as f:
            f.write(geometry.to_xyz(atoms))
        return g.BasisSet(GBS, path)


def _molecule(case, seed):
    """The case's molecule; its random placements and the seed's displacements."""
    return _atoms(case["mol"], case["size"], case["stretch"], np.random.default_rng([11, seed]))


def _batch_molecules(case, seed):
    """Alkanes and water clusters of up to `largest` carbons or monomers."""
    rng = np.random.default_rng([7, case["count"], case["largest"]])
    sizes = rng.integers(1, case["largest"] + 1, size=case["count"])
    move = np.random.default_rng([13, seed])
    return [_atoms("alkane" if k < case["count"] // 2 else "water", int(s), case["stretch"], move)
            for k, s in enumerate(sizes)]


def _density(atoms, seed):
    """A symmetric matrix with a density's sizes: about half an electron pair
    on the diagonal, falling off with the distance of the centres."""
    shells, _ = _shells(atoms)
    centre = np.concatenate([np.repeat(s["x"][None], 2 * s["l"] + 1, 0) for s in shells])
    n = len(centre)
    a = np.random.default_rng([17, seed]).normal(size=(n, n))
    r = np.sqrt(((centre[:, None] - centre[None]) ** 2).sum(-1))
    d = 0.2 * (a + a.T) * np.exp(-r / 2.5)
    d[np.arange(n), np.arange(n)] += 0.5
    return d


def _spectrum(n, nocc, seed):
    """A Fock matrix of the orthogonal basis with a closed-shell molecule's
    levels (core, valence, gap, virtuals), and a symmetric S^-1/2."""
    gen = torch.Generator().manual_seed(int(seed) + 1000003)
    core = max(1, nocc // 4)
    e = torch.cat([-11.0 - torch.rand(core, generator=gen, dtype=torch.float64),
                   -1.2 + 0.8 * torch.rand(nocc - core, generator=gen, dtype=torch.float64),
                   0.15 + 3.5 * torch.rand(n - nocc, generator=gen, dtype=torch.float64) ** 2])
    s = torch.exp(torch.empty(n, dtype=torch.float64).uniform_(math.log(1e-3), math.log(6.0), generator=gen))
    a, b = (torch.randn(n, n, generator=gen, dtype=torch.float64) for _ in range(2))
    qa, qb = (torch.linalg.qr(m.to(_device()))[0].cpu() for m in (a, b))
    f = (qa * e) @ qa.T
    x = (qb * s.rsqrt()) @ qb.T
    return (0.5 * (f + f.T)).numpy(), (0.5 * (x + x.T)).numpy()


def _quartets(case, nshells):
    return np.random.default_rng([19, case["nquartets"]]).integers(0, nshells, size=(case["nquartets"], 4)).astype(np.int32)


# ---- the calls ------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("batch", "scf"):
        mols = _batch_molecules(case, seed)
        batch = g.Batch([_basis(a) for a in mols])
        if kind == "scf":
            return dict(case=case, batch=batch)
        return dict(case=case, batch=batch, D=[_density(a, seed + 31 * k) for k, a in enumerate(mols)])
    atoms = _molecule(case, seed)
    basis = _basis(atoms)
    state = dict(case=case, basis=basis)
    if kind == "fock":
        state["pf"] = g.PFock(basis, max_numdmat=case["nden"])
        if case["tau"] > 0:
            state["pf"].set_precision(case["tau"])
        state["D"] = [_density(atoms, seed + 31 * k) for k in range(case["nden"])]
    elif kind == "purify":
        state["pu"] = g.Purif(basis)
        state["F"], X = _spectrum(basis.nbf, basis.nocc, seed)
        state["pu"].set_xs(X, np.eye(basis.nbf))
    elif kind == "eri":
        state["erd"] = g.ERD(basis)
        state["q"] = _quartets(case, basis.nshells)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fock":
        pf = state["pf"]
        for k, D in enumerate(state["D"]):
            pf.put_den_mat(D, k)
        pf.commit()
        pf.compute_fock()
        return [pf.get_mat(g.MAT_F, k) for k in range(len(state["D"]))]
    if kind == "batch":
        return np.concatenate([F.reshape(-1) for F in state["batch"].fock(state["D"])])
    if kind == "scf":
        b = state["batch"]
        energy, _ = b.scf(max_iters=case["iters"], ediff=1e-30)
        return dict(energy=energy, density=np.concatenate([D.reshape(-1) for D in b.get_density()]))
    if kind == "purify":
        return state["pu"].purify(state["F"])[0]
    if kind == "eri":
        return state["erd"].quartets(state["q"])[0].base
    pf = g.PFock(state["basis"])
    S, X, H = pf.overlap(), pf.x_matrix(), pf.core_hamiltonian()
    pf.close()
    return dict(S=S, X=X, H=H)


# ---- the work that no method can leave out -----------------------------------------


def _counts(atoms):
    """Functions, function pairs that overlap, primitive pairs in them."""
    shells, _ = _shells(atoms)
    n = sum(2 * s["l"] + 1 for s in shells)
    pairs = prims = 0
    for i, a in enumerate(shells):
        for b in shells[: i + 1]:
            r2 = float(((a["x"] - b["x"]) ** 2).sum())
            mu = a["a"].min() * b["a"].min() / (a["a"].min() + b["a"].min())
            if mu * r2 < 23.0:  # e^-23: products below the screening threshold
                pairs += (2 * a["l"] + 1) * (2 * b["l"] + 1)
                prims += len(a["a"]) * len(b["a"])
    return n, pairs, prims


def _fock_flops(atoms, nden):
    """Unique integrals of overlapping pairs, about 60 operations each to form
    and 12 to digest; the contraction degree raises the first."""
    n, pairs, prims = _counts(atoms)
    unique = 0.5 * pairs * pairs
    return unique * (20.0 * max(1.0, (prims / pairs) ** 2) + 12.0 * nden)


def work(case):
    kind = case["kind"]
    if kind in ("batch", "scf"):
        mols = _batch_molecules(case, 1)
        nn = [sum(2 * s["l"] + 1 for s in _shells(a)[0]) for a in mols]
        builds = case["iters"] if kind == "scf" else 1
        flops = builds * sum(_fock_flops(a, 1) for a in mols)
        if kind == "scf":
            flops += builds * sum(40.0 * 2 * n ** 3 for n in nn)
        return dict(bytes=16.0 * sum(n * n for n in nn), flops=flops)
    atoms = _molecule(case, 1)
    n, pairs, prims = _counts(atoms)
    if kind == "fock":
        return dict(bytes=16.0 * n * n * case["nden"], flops=_fock_flops(atoms, case["nden"]))
    if kind == "purify":
        # about 40 iterations of two products of symmetric matrices, then X D X
        return dict(bytes=24.0 * n * n, flops=82.0 * n ** 3)
    if kind == "eri":
        mean = (n / len(_shells(atoms)[0])) ** 4
        return dict(bytes=case["nquartets"] * (16.0 + 8.0 * mean), flops=case["nquartets"] * mean * 60.0)
    # the eigenvalue problem of S and the nuclear attraction integrals
    return dict(bytes=24.0 * n * n, flops=9.0 * n ** 3 + 40.0 * prims * len(atoms))


# ---- the same values in plain torch and numpy, 64 bits --------------------------------
# McMurchie and Davidson, J. Comput. Phys. 26, 218 (1978): Hermite expansions
# of the primitive pairs and Hermite Coulomb integrals.


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


_ELEMENTS = {}


def _element(symbol):
    """[(l, [(exponent, coefficient), ...]), ...] of one element of the basis file."""
    if not _ELEMENTS:
        cur, left = None, 0
        for line in open(GBS):
            t = line.split()
            if left:
                cur[-1][1].append((float(t[0]), float(t[1])))
                left -= 1
            elif len(t) == 2 and t[1] == "0":
                cur = _ELEMENTS.setdefault(t[0], [])
            elif len(t) == 3 and t[0] in "SPD":
                cur.append(("SPD".index(t[0]), []))
                left = int(t[1])
    return _ELEMENTS[symbol]


def _shells(atoms):
    """Normalised contracted shells in atom order, and the nuclei."""
    out = []
    for symbol, x in atoms:
        for l, prims in _element(symbol):
            a = np.array([p[0] for p in prims])
            odd = (1, 1, 3)[l]
            c = np.array([p[1] for p in prims]) * np.sqrt((4 * a) ** l * (2 * a / math.pi) ** 1.5 / odd)
            p = a[:, None] + a[None]
            c = c / math.sqrt((c[:, None] * c[None] * odd / (2 * p) ** l * (math.pi / p) ** 1.5).sum())
            out.append(dict(l=l, a=a, c=c, x=np.array(x) * BOHR))
    return out, [(CHARGE[s], np.array(x) * BOHR) for s, x in atoms]


def _cartesian(l):
    return [(i, l - i - k, k) for i in range(l, -1, -1) for k in range(l - i + 1)]


def _spherical(l):
    r3 = math.sqrt(3.0)
    rows = {0: [[1.0]], 1: np.eye(3).tolist(),
            2: [[0, r3, 0, 0, 0, 0], [0, 0, 0, 0, r3, 0], [-0.5, 0, 0, -0.5, 0, 1.0], [0, 0, r3, 0, 0, 0],
                [0.5 * r3, 0, 0, -0.5 * r3, 0, 0]]}
    return torch.tensor(rows[l], dtype=torch.float64, device=_device())


def _hermite_1d(la, lb, a, b, ab):
    """E[i][j][t] of one dimension, for arrays of primitive pairs."""
    p, zero = a + b, torch.zeros_like(a)
    E = {(0, 0): [torch.exp(-a * b / p * ab * ab)]}

    def up(e, shift):
        get = lambda t: e[t] if 0 <= t < len(e) else zero  # noqa: E731
        return [get(t - 1) / (2 * p) + shift * get(t) + (t + 1) * get(t + 1) for t in range(len(e) + 1)]

    for i in range(la + 1):
        if i:
            E[i, 0] = up(E[i - 1, 0], -b / p * ab)
        for j in range(1, lb + 1):
            E[i, j] = up(E[i, j - 1], a / p * ab)
    return E


def _hermites(L):
    return [(t, u, v) for k in range(L + 1) for t in range(k, -1, -1) for u in range(k - t, -1, -1)
            for v in [k - t - u]]


class _Pairs:
    """All primitive pairs of the shell pairs (i, j) of one angular type, l_i
    >= l_j: exponents p, centres P, Hermite coefficients E[pair, component,
    tuv] with the contraction in them, and the owning shell pair."""

    def __init__(self, shells, la, lb):
        self.la, self.lb, self.list = la, lb, []
        cols = []
        for i, j in itertools.product(range(len(shells)), repeat=2):
            A, B = shells[i], shells[j]
            if A["l"] != la or B["l"] != lb or (la == lb and j > i):
                continue
            for (x, cx), (y, cy) in itertools.product(zip(A["a"], A["c"]), zip(B["a"], B["c"])):
                cols.append([x, y, cx * cy, len(self.list), *A["x"], *B["x"]])
            self.list.append((i, j))
        t = torch.tensor(np.array(cols).reshape(-1, 10), dtype=torch.float64, device=_device())
        self.a, self.b, self.c, self.own = t[:, 0], t[:, 1], t[:, 2], t[:, 3].long()
        self.A, self.B = t[:, 4:7], t[:, 7:10]
        self.p = self.a + self.b
        self.P = (self.a[:, None] * self.A + self.b[:, None] * self.B) / self.p[:, None]
        self.E1 = [_hermite_1d(la, lb + 2, self.a, self.b, self.A[:, d] - self.B[:, d]) for d in range(3)]
        self.tuv = _hermites(la + lb)

        def block(ca, cb):
            ex, ey, ez = (self.E1[d][ca[d], cb[d]] for d in range(3))
            zero = torch.zeros_like(self.a)
            return torch.stack([self.c * ex[t] * ey[u] * ez[v] if t < len(ex) and u < len(ey) and v < len(ez)
                                else zero for t, u, v in self.tuv], 1)

        self.E = self.transform(block)  # [prim, component, tuv]

    def transform(self, block):
        """block(cartesian a, cartesian b) -> [prim, k] to spherical [prim, component, k]."""
        m = torch.stack([torch.stack([block(ca, cb) for cb in _cartesian(self.lb)], 1) for ca in _cartesian(self.la)], 1)
        m = torch.einsum("ai,bj,pijk->pabk", _spherical(self.la), _spherical(self.lb), m)
        return m.reshape(len(self.a), -1, m.shape[-1])


def _pair_types(shells):
    got = [_Pairs(shells, la, lb) for la in range(3) for lb in range(la + 1)]
    return [p for p in got if p.list]


_GRID = None


def _boys(M, T):
    """F_0 .. F_M(T): Taylor series on a grid of step 1/16 up to 40, the
    recursions downwards there and upwards beyond."""
    global _GRID
    if _GRID is None or _GRID.device != T.device:
        t = np.arange(0, 16 * 40 + 2, dtype=np.longdouble) / 16
        cols = []
        for m in range(24):
            term = 1 / np.longdouble(2 * m + 1) + 0 * t
            s = term.copy()
            for k in range(1, 260):
                term = term * 2 * t / (2 * m + 2 * k + 1)
                s += term
            cols.append(np.exp(-t) * s)
        _GRID = torch.tensor(np.array(cols).astype(np.float64), device=T.device)
    Ts = T.clamp(max=40.0)
    i = (Ts * 16 + 0.5).long()
    d = i.to(T.dtype) / 16 - Ts
    f, w = torch.zeros_like(T), torch.ones_like(T)
    for k in range(12):
        f += _GRID[M + k][i] * w
        w = w * d / (k + 1)
    e = torch.exp(-T)
    low = [f]
    for m in range(M - 1, -1, -1):
        low.insert(0, (2 * T * low[0] + e) / (2 * m + 1))
    high = [0.5 * torch.sqrt(math.pi / T.clamp(min=1.0))]
    for m in range(M):
        high.append(((2 * m + 1) * high[-1] - e) / (2 * T.clamp(min=1.0)))
    return [torch.where(T < 40.0, x, y) for x, y in zip(low, high)]


def _coulomb(L, alpha, X):
    """R_tuv for t + u + v <= L: {(t, u, v): array}; X: the three distances."""
    F = _boys(L, alpha * (X[0] ** 2 + X[1] ** 2 + X[2] ** 2))
    R = {}
    for n in range(L, -1, -1):
        S = {(0, 0, 0): (-2 * alpha) ** n * F[n]}
        for h in _hermites(L - n)[1:]:
            d = next(k for k in range(3) if h[k])
            one = tuple(v - (k == d) for k, v in enumerate(h))
            two = tuple(v - 2 * (k == d) for k, v in enumerate(h))
            S[h] = X[d] * R[one] + ((h[d] - 1) * R[two] if h[d] > 1 else 0.0)
        R = S
    return R


def _eri_block(bra, ket, at=slice(None)):
    """Integrals [bra pair, bra component, ket pair, ket component] of the bra primitives `at`."""
    L = bra.la + bra.lb + ket.la + ket.lb
    p, q = bra.p[at, None], ket.p[None]
    alpha = p * q / (p + q)
    R = _coulomb(L, alpha, [bra.P[at, d][:, None] - ket.P[None, :, d] for d in range(3)])
    pref = 2 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q))
    nk = len(ket.list)
    out = torch.zeros(len(bra.list), bra.E.shape[1], nk, ket.E.shape[1], dtype=torch.float64, device=p.device)
    for h1, (t, u, v) in enumerate(bra.tuv):
        y = sum((-1) ** sum(h) * (R[t + h[0], u + h[1], v + h[2]] * pref)[:, :, None] * ket.E[None, :, :, k]
                for k, h in enumerate(ket.tuv))
        z = torch.zeros(y.shape[0], nk, y.shape[2], dtype=y.dtype, device=y.device).index_add_(1, ket.own, y)
        e = bra.E[at, :, h1]
        out.index_add_(0, bra.own[at], e[:, :, None, None] * z[:, None])
    return out


def _tensor(shells):
    """All (mn|pq)."""
    start = np.concatenate([[0], np.cumsum([2 * s["l"] + 1 for s in shells])]).astype(int)
    n, dev = int(start[-1]), _device()
    types = _pair_types(shells)
    where = torch.zeros(n, n, dtype=torch.long, device=dev)  # function pair -> row of the pair matrix
    at, base = 0, []
    for t in types:
        base.append(at)
        for i, j in t.list:
            na, nb = 2 * t.la + 1, 2 * t.lb + 1
            rows = at + torch.arange(na * nb, device=dev).reshape(na, nb)
            where[start[i]:start[i] + na, start[j]:start[j] + nb] = rows
            where[start[j]:start[j] + nb, start[i]:start[i] + na] = rows.T
            at += na * nb
    G = torch.zeros(at, at, dtype=torch.float64, device=dev)
    for x, bra in enumerate(types):
        for y, ket in enumerate(types[: x + 1]):
            block = torch.zeros(len(bra.list), bra.E.shape[1], len(ket.list), ket.E.shape[1], dtype=torch.float64,
                                device=dev)
            cells = len(ket.p) * len(_hermites(bra.la + bra.lb + ket.la + ket.lb))
            step = max(1, int(4e7 / cells))
            for k in range(0, len(bra.p), step):
                block += _eri_block(bra, ket, slice(k, k + step))
            nb, nk = block.shape[0] * block.shape[1], block.shape[2] * block.shape[3]
            G[base[x]:base[x] + nb, base[y]:base[y] + nk] = block.reshape(nb, nk)
            G[base[y]:base[y] + nk, base[x]:base[x] + nb] = block.reshape(nb, nk).T
    flat = where.reshape(-1)
    return G[flat][:, flat].reshape(n, n, n, n)


def _exact_fock(shells, densities):
    I = _tensor(shells)
    n = I.shape[0]
    swapped = I.permute(0, 2, 1, 3).reshape(n * n, n * n)
    out = []
    for D in densities:
        d = torch.tensor(D, device=I.device).reshape(-1)
        out.append((2 * (I.reshape(n * n, n * n) @ d) - swapped @ d).reshape(n, n).cpu().numpy())
    return out


def _exact_one(shells, nuclei):
    """Overlap, S^-1/2 and core Hamiltonian."""
    start = np.concatenate([[0], np.cumsum([2 * s["l"] + 1 for s in shells])]).astype(int)
    n = int(start[-1])
    S, H = np.zeros((n, n)), np.zeros((n, n))
    for t in _pair_types(shells):
        s1 = lambda d, i, j: t.E1[d][i, j][0] * torch.sqrt(math.pi / t.p) if j >= 0 else 0.0  # noqa: E731

        def t1(d, i, j):
            return (-2 * t.b ** 2 * s1(d, i, j + 2) + t.b * (2 * j + 1) * s1(d, i, j)
                    - 0.5 * j * (j - 1) * s1(d, i, j - 2))

        def block(ca, cb):
            s = [s1(d, ca[d], cb[d]) for d in range(3)]
            k = [t1(d, ca[d], cb[d]) for d in range(3)]
            return torch.stack([t.c * s[0] * s[1] * s[2],
                                t.c * (k[0] * s[1] * s[2] + s[0] * k[1] * s[2] + s[0] * s[1] * k[2])], 1)

        ST = t.transform(block)
        V = torch.zeros_like(ST[:, :, 0])
        for z, x in nuclei:
            R = _coulomb(t.la + t.lb, t.p, [t.P[:, d] - x[d] for d in range(3)])
            V -= z * (2 * math.pi / t.p)[:, None] * sum(t.E[:, :, k] * R[h][:, None] for k, h in enumerate(t.tuv))
        vals = torch.stack([ST[:, :, 0], ST[:, :, 1] + V], 2)
        vals = torch.zeros(len(t.list), *vals.shape[1:], dtype=vals.dtype, device=vals.device).index_add_(0, t.own, vals)
        na, nb = 2 * t.la + 1, 2 * t.lb + 1
        vals = vals.reshape(len(t.list), na, nb, 2).cpu().numpy()
        for (i, j), v in zip(t.list, vals):
            for k, M in enumerate((S, H)):
                M[start[i]:start[i] + na, start[j]:start[j] + nb] = v[:, :, k]
                M[start[j]:start[j] + nb, start[i]:start[i] + na] = v[:, :, k].T
    w, U = np.linalg.eigh(S)
    return dict(S=S, X=(U / np.sqrt(w)) @ U.T, H=H)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "scf"):
        return None
    atoms = _molecule(case, seed)
    shells, nuclei = _shells(atoms)
    n = sum(2 * s["l"] + 1 for s in shells)
    if kind == "fock":
        if n > 150:  # the n^4 integrals take longer than the check allows
            return None
        return _exact_fock(shells, [_density(atoms, seed + 31 * k) for k in range(case["nden"])])
    if kind == "purify":
        nocc = sum(z for z, _ in nuclei) // 2
        F, X = _spectrum(n, nocc, seed)
        _, U = np.linalg.eigh(F)
        XU = X @ U[:, :nocc]
        return XU @ XU.T
    if kind == "setup":
        return _exact_one(shells, nuclei)
    if n > 150:
        return None
    I = _tensor(shells)
    start = np.concatenate([[0], np.cumsum([2 * s["l"] + 1 for s in shells])]).astype(int)
    size = np.array([2 * s["l"] + 1 for s in shells])
    at = []
    for M, N, P, Q in _quartets(case, len(shells)):
        m, nn, p, q = (np.arange(start[k], start[k] + size[k]) for k in (M, N, P, Q))
        # first index fastest
        at.append((((m[None, None, None, :] * n + nn[None, None, :, None]) * n + p[None, :, None, None]) * n
                   + q[:, None, None, None]).reshape(-1))
    return I.reshape(-1)[torch.from_numpy(np.concatenate(at)).to(I.device)].cpu().numpy()
