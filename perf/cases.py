"""Cases that stand for the work this package does in a quantum chemistry program: direct Coulomb
and exchange builds through the public entry points (IntBox.coulomb / exchange and their
device-pointer forms, JKBatch), their nuclear gradients, and the one-electron integrals.

A case is a dict of plain values:
  kind      "jk": one SCF iteration's J and K over a symmetric pair list;
            "transition": J and K of a transition density (not symmetric, so D24symm is off);
            "fragments": J and exchange of one fragment in the density of another, in two basis
            sets (rectangular lists);
            "gradient": the nuclear gradient of the Coulomb and the exchange energy;
            "one_electron": overlap, kinetic energy and nuclear attraction;
            "batch": J and K of many independent molecules in one call.
  system, n the molecule: "water" (a random cluster of n waters, 6-31G* and the like) or "alkane"
            (C_n H_2n+2); for a batch, clusters of 1 to `largest` waters.
  density   "projector": the dense projector of the benchmark and the tests (no decay: an early
            iteration); "local": a density matrix that decays with distance, as a converged SCF
            of an insulator has.
  api       "host": Tensors in and out; "device": the caller's own HBM buffers.
  thresp, thredp, omega  the sieve, the FP32 route (thredp > thresp) and the range separation of K.

prepare() makes the molecule, the density and the pair list from the seed; run() is one pass.
exact() computes the same results in FP64 with torch, from a Hermite expansion of all function
pairs without any screening, for the sizes where that takes a few seconds.
"""
import math

import numpy as np
import torch

import lightspeed_amd as ls
from lightspeed_amd import workloads as W

THRE = 1.0e-12


def listed():
    base = {"system": "water", "density": "local", "api": "device", "thresp": THRE, "thredp": THRE, "omega": 0.0}

    def case(name, **kw):
        return dict(base, name=name, **kw)

    return [
        # the smallest molecule in the smallest basis: what a call costs beside its integrals
        case("water1_sto3g", kind="jk", n=1, basis="sto-3g", density="projector", api="host"),
        # an ordinary small SCF (the tests' own cluster)
        case("water10_631g", kind="jk", n=10, basis="6-31g", density="projector", api="host"),
        # a chain in a spherical basis, through the host API (pure <-> Cartesian transforms included)
        case("alkane20_ccpvdz", kind="jk", system="alkane", n=20, basis="cc-pvdz", density="projector", api="host"),
        # the benchmark's cluster and basis, first iterations: a dense density
        case("water64_631gss", kind="jk", n=64, basis="6-31gss", density="projector"),
        # the same on the mixed route, near convergence
        case("water64_631gss_mixed", kind="jk", n=64, basis="6-31gss", thredp=1.0e-6),
        # a large cluster near convergence
        case("water128_631gs", kind="jk", n=128, basis="6-31gs"),
        # a range-separated hybrid functional: K of c/r + (1 - c) erf(omega r)/r
        case("water24_631gss_range", kind="jk", n=24, basis="6-31gss", omega=0.3),
        # an excited-state iteration (transition density)
        case("water17_631gs_transition", kind="transition", n=17, basis="6-31gs"),
        # one fragment in the field of another, different bases
        case("water12_in_water19", kind="fragments", n=12, basis="6-31gss", n_other=19, basis_other="6-31g",
             api="host"),
        # one geometry step's two-electron gradient
        case("water8_631gs_gradient", kind="gradient", n=8, basis="6-31gs", api="host"),
        # the start of an SCF
        case("water48_631gss_one_electron", kind="one_electron", n=48, basis="6-31gss", api="host"),
        # many small molecules (a screening run, or one step of an ensemble)
        case("batch60_631gs", kind="batch", n=60, largest=16, basis="6-31gs", density="projector"),
    ]


def draw(rng):
    def logint(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.499)))))))

    c = {"kind": rng.choice(["jk", "jk", "jk", "jk", "jk", "transition", "fragments", "gradient", "one_electron",
                             "batch"]),
         "system": "water", "density": rng.choice(["local", "local", "projector"]),
         "api": rng.choice(["host", "device"]), "thresp": rng.choice([1.0e-12, 1.0e-12, 1.0e-11, 1.0e-10]),
         "omega": 0.0}
    c["thredp"] = c["thresp"]
    bases = ["sto-3g", "6-31g", "6-31gs", "6-31gss", "cc-pvdz"]
    if c["kind"] == "jk":
        c["basis"] = rng.choice(bases)
        if rng.random() < 0.25:
            c["system"], c["n"] = "alkane", logint(2, 19)
        else:
            c["n"] = logint(1, 40 if c["basis"] == "cc-pvdz" else 90)
        if rng.random() < 0.3:
            c["thredp"] = 1.0e-6
        elif rng.random() < 0.3:
            c["omega"] = rng.choice([0.11, 0.3, 0.4])
    elif c["kind"] == "transition":
        c["basis"], c["n"] = rng.choice(bases[1:4]), logint(2, 32)
    elif c["kind"] == "fragments":
        c.update(basis=rng.choice(bases[:4]), basis_other=rng.choice(bases[:4]), n=logint(1, 30), n_other=logint(1, 30),
                 api="host")
    elif c["kind"] == "gradient":
        c.update(basis=rng.choice(bases[:3]), n=logint(1, 8), api="host", density="local")
    elif c["kind"] == "one_electron":
        c.update(basis=rng.choice(bases[:4]), n=logint(1, 90), api="host")
    else:
        c.update(basis=rng.choice(bases[1:4]), n=logint(3, 64), largest=rng.randint(2, 14), api="device")
    return c


# ---------------------------------------------------------------- inputs


def _molecule(system, n, seed):
    if system == "water":
        return W.water_cluster(n, W.water_cluster_box(n), 1000 + seed)
    mol = W.alkane(n)
    shift = np.random.default_rng(seed).normal(0.0, 0.03, (mol.natom, 3))  # bohr: thermal displacements
    atoms = [a._replace(x=a.x + s[0], y=a.y + s[1], z=a.z + s[2]) for a, s in zip(mol.atoms, shift)]
    return ls.Molecule(mol.name, atoms)


def _nocc(mol):
    return int(sum(a.Z for a in mol.atoms)) // 2


def _orbitals(bas, nocc, density, seed):
    """Orthonormal columns, nao x nocc: dense, or each decaying from an atom of its own."""
    rng = np.random.default_rng(seed + 77)
    A = rng.standard_normal((bas.nao, nocc))
    if density == "local":
        at = np.zeros(bas.nao, dtype=int)
        xyz = {}
        for p in bas.primitives:
            at[p.aoIdx:p.aoIdx + (2 * p.L + 1 if p.is_pure else p.ncart)] = p.atomIdx
            xyz[p.atomIdx] = (p.x, p.y, p.z)
        X = np.array([xyz[k] for k in range(len(xyz))])
        own = np.linspace(0, bas.nao - 1, nocc).astype(int)  # every orbital has a function of its own
        r = np.linalg.norm(X[at][:, None, :] - X[at[own]][None, :, :], axis=2)
        A *= np.exp(-r / 1.3)
        A[own, np.arange(nocc)] = 3.0
        L = np.linalg.cholesky(A.T @ A)
        return np.linalg.solve(L, A.T).T
    return np.linalg.qr(A)[0]


def _density(bas, nocc, density, seed):
    C = _orbitals(bas, nocc, density, seed)
    return np.ascontiguousarray(C @ C.T)


def _operators(case):
    """The operators of J and of K."""
    J = ([1.0], [-1.0])
    return J, (([0.2, 0.8], [-1.0, case["omega"]]) if case["omega"] else J)


def _inputs(case, seed):
    """Molecules, bases and host densities of a case (kind-dependent), from the seed alone."""
    if case["kind"] == "batch":
        sizes = np.random.default_rng(case["n"]).integers(1, case["largest"] + 1, size=case["n"])
        out = []
        for i, n in enumerate(sizes):
            mol = _molecule("water", int(n), 1000 * seed + i)
            bas = ls.Basis.from_gbs_file(mol, case["basis"])
            out.append((mol, bas, _density(bas, _nocc(mol), case["density"], 1000 * seed + i)))
        return out
    mol = _molecule(case["system"], case["n"], seed)
    bas = ls.Basis.from_gbs_file(mol, case["basis"])
    if case["kind"] == "transition":
        no = _nocc(mol)
        C = _orbitals(bas, no, case["density"], seed)
        V = _orbitals(bas, no, case["density"], seed + 1)
        amp = np.random.default_rng(seed + 5).standard_normal(no) / math.sqrt(no)
        return mol, bas, np.ascontiguousarray((C * amp) @ V.T)
    D = _density(bas, _nocc(mol), case["density"], seed)
    if case["kind"] != "fragments":
        return mol, bas, D
    other = _molecule("water", case["n_other"], seed + 500)
    # the second fragment beside the first: 2 angstrom between their extents along x
    gap = max(a.x for a in mol.atoms) - min(a.x for a in other.atoms) + 2.0 * ls.BOHR_PER_ANG
    other = ls.Molecule("other", [a._replace(x=a.x + gap) for a in other.atoms])
    bas2 = ls.Basis.from_gbs_file(other, case["basis_other"])
    return mol, bas, bas2, _density(bas2, _nocc(other), case["density"], seed + 1)


def _cartesian(bas, D):
    return np.array(ls.PureTransform.pureToCart2(bas, bas, ls.Tensor.array(D)).np) if bas.has_pure else D


def _pairs(b1, b2, case):
    return ls.PairList.build_schwarz(b1, b2, b1 is b2, case["thresp"])


def prepare(case, seed):
    opJ, opK = _operators(case)
    s = {"case": case, "res": ls.ResourceList.build(), "opJ": ls.Ewald(*opJ), "opK": ls.Ewald(*opK)}
    inp = _inputs(case, seed)
    if case["kind"] == "batch":
        s["batch"] = b = ls.JKBatch.build(s["res"], [_pairs(bas, bas, case) for _, bas, _ in inp])
        flat = np.zeros(b.nelem)
        for off, (_, bas, D) in zip(b.offsets, inp):
            n = bas.ncart
            np.lib.stride_tricks.as_strided(flat[off:], (n, n), (8 * b.ld, 8))[:] = _cartesian(bas, D)
        s["D"] = torch.from_numpy(flat).cuda()
        s["J"], s["K"] = torch.empty_like(s["D"]), torch.empty_like(s["D"])
        return s
    mol, bas = inp[0], inp[1]
    s["pairs"] = _pairs(bas, bas, case)
    if case["kind"] == "one_electron":
        s["charges"] = ls.Tensor.array(np.ascontiguousarray(mol.xyzZ, dtype=float))
    elif case["kind"] == "fragments":
        s["other"], s["cross"] = _pairs(inp[2], inp[2], case), _pairs(bas, inp[2], case)
        s["D"] = ls.Tensor.array(inp[3])
    elif case["api"] == "host":
        s["D"] = ls.Tensor.array(inp[2])
    else:
        s["D"] = torch.from_numpy(_cartesian(bas, inp[2])).cuda()
        s["J"], s["K"] = torch.empty_like(s["D"]), torch.empty_like(s["D"])
    return s


def run(state):
    s = state
    c, I = s["case"], ls.IntBox
    t, td = c["thresp"], c["thredp"]
    if c["kind"] == "one_electron":
        p = s["pairs"]
        return {"S": I.overlap(s["res"], p).np, "T": I.kinetic(s["res"], p).np,
                "V": I.potential(s["res"], s["opJ"], p, s["charges"]).np}
    if c["kind"] == "gradient":
        return {"J": I.coulombGrad(s["res"], s["opJ"], s["pairs"], s["D"], s["D"], t, td).np,
                "K": I.exchangeGrad(s["res"], s["opJ"], s["pairs"], s["D"], s["D"], True, True, True, t, td).np}
    if c["kind"] == "fragments":
        return {"J": I.coulomb(s["res"], s["opJ"], s["pairs"], s["other"], s["D"], t, td).np,
                "K": I.exchange(s["res"], s["opJ"], s["cross"], s["cross"], s["D"], True, t, td).np}
    symm = c["kind"] != "transition"
    if c["api"] == "host" and c["kind"] != "batch":
        p = s["pairs"]
        return {"J": I.coulomb(s["res"], s["opJ"], p, p, s["D"], t, td).np,
                "K": I.exchange(s["res"], s["opK"], p, p, s["D"], symm, t, td).np}
    s["J"].zero_()
    s["K"].zero_()
    # the builds run on the library's own stream and return when they are done: torch's part before
    # them has to be done as well
    torch.cuda.current_stream().synchronize()
    if c["kind"] == "batch":
        s["batch"].jk_device(s["opJ"], s["D"].data_ptr(), t, td, s["J"].data_ptr(), s["K"].data_ptr())
    else:
        p = s["pairs"]
        I.coulomb_device(s["opJ"], p, p, s["D"].data_ptr(), t, td, s["J"].data_ptr())
        I.exchange_device(s["opK"], p, p, s["D"].data_ptr(), symm, t, td, s["K"].data_ptr())
    return {"J": s["J"], "K": s["K"]}


# ---------------------------------------------------------------- work


def _quartet_flops(L1, L2, L3, L4):
    """Rys quadrature with the 2-D recurrences: roots, one-dimensional integrals, assembly."""
    nc = [(L + 1) * (L + 2) // 2 for L in (L1, L2, L3, L4)]
    nr, pi, g = (L1 + L2 + L3 + L4) // 2 + 1, nc[0] * nc[1] * nc[2] * nc[3], (L1 + L2 + 1) * (L3 + L4 + 1)
    return 40 + nr * (30 + 9 * g + 3 * pi) + 2 * pi


def work(case):
    """Bytes: densities, pair data (a centre, exponents, a prefactor and a bound each) and results,
    once.  Flops: the primitive quartets that the sieve leaves, at the count above (for gradients
    at one quantum more on the three centres that are differentiated)."""
    c, inp = case, _inputs(case, 0)
    if c["kind"] == "one_electron":
        p = _pairs(inp[1], inp[1], c)
        per = sum(l.npair * _quartet_flops(l.L1, l.L2, 0, 0) for l in p.pairlists)
        return {"bytes": 3 * 8 * inp[1].nao ** 2 + 64 * p.npair, "flops": per * inp[0].natom}
    ls.hip_init(0)

    def up(x):
        d = ls.DeviceArray(list(x.shape))
        d.upload(x)
        return d

    def count(pl12, pl34, D, symm, grad=0):
        d = up(D)
        nj, nk = ls.count_quartets(pl12, pl34, d.ptr, d.ptr, symm, c["thresp"])
        f = np.array([_quartet_flops(i // 125 + grad, i // 25 % 5 + grad, i // 5 % 5 + grad, i % 5) for i in range(625)])
        return float(nj @ f), float(nk @ f)

    if c["kind"] == "batch":
        b = fl = 0.0
        for _, bas, D in inp:
            p = _pairs(bas, bas, c)
            fl += sum(count(p, p, _cartesian(bas, D), True))
            b += 24 * bas.ncart ** 2 + 64 * p.npair
        return {"bytes": b, "flops": fl}
    if c["kind"] == "fragments":
        p, o, x = _pairs(inp[1], inp[1], c), _pairs(inp[2], inp[2], c), _pairs(inp[1], inp[2], c)
        n1, n2 = inp[1].nao, inp[2].nao
        # J pairs the fragments' own lists; K runs over the pairs that join them
        D = _cartesian(inp[2], inp[3])
        fj = sum(a.npair * b.npair * _quartet_flops(a.L1, a.L2, b.L1, b.L2) for a in p.pairlists for b in o.pairlists)
        return {"bytes": 8 * (2 * n1 * n1 + 2 * n2 * n2) + 64 * (p.npair + o.npair + x.npair),
                "flops": fj + count(x, x, D, True)[1]}
    bas, D = inp[1], _cartesian(inp[1], inp[2])
    p = _pairs(bas, bas, c)
    symm = c["kind"] != "transition"
    fl = sum(count(p, p, D, symm, 1 if c["kind"] == "gradient" else 0))
    out = 2 * 8 * bas.nao ** 2 if c["kind"] != "gradient" else 0
    return {"bytes": 8 * bas.nao ** 2 + out + 64 * p.npair, "flops": fl}


# ---------------------------------------------------------------- the same results in FP64
#
# (ab|O|cd) = sum_tu E^ab_t E^cd_u (-1)^|u| R_{t+u}(P - Q) over the primitive pairs, McMurchie and
# Davidson, J. Comput. Phys. 26, 218 (1978); R from the Boys functions, which come from their
# Taylor expansions about a grid (power series at the grid points) and their large-T limit.


def _powers(L):
    return [(L - i, i - j, j) for i in range(L + 1) for j in range(i + 1)]


def _hermites(L):
    return [t for k in range(L + 1) for t in _powers(k)]


_BOYS = {}


def _boys(N, T):
    """F_0 .. F_N at T."""
    dev, step, top, terms = T.device, 1.0 / 16, 64.0, 9
    if dev not in _BOYS:
        g = torch.arange(0, top + 2 * step, step, dtype=torch.float64, device=dev)
        M = 30
        s = t = torch.full_like(g, 1.0 / (2 * M + 1))
        for k in range(1, 300):
            t = t * 2 * g / (2 * M + 2 * k + 1)
            s = s + t
        F = [torch.exp(-g) * s]
        for n in range(M - 1, -1, -1):
            F.append((2 * g * F[-1] + torch.exp(-g)) / (2 * n + 1))
        _BOYS[dev] = torch.stack(F[::-1])
    tab = _BOYS[dev]
    small = T < top
    Ts = torch.where(small, T, torch.zeros_like(T))
    i = (Ts / step + 0.5).long()
    h = i * step - Ts
    Tl = torch.where(small, torch.full_like(T, top), T)
    out = []
    large = 0.5 * torch.sqrt(math.pi / Tl)
    for n in range(N + 1):
        f = tab[n + terms][i] / terms * h
        for k in range(terms - 1, 0, -1):
            f = (tab[n + k][i] + f) * h / k
        out.append(torch.where(small, tab[n][i] + f, large))
        large = large * (2 * n + 1) / (2 * Tl)
    return out


def _hermite_R(L, alpha, X, op):
    """R_t, |t| <= L, for exponents alpha and distances X (..., 3) under the operator `op`."""
    T = alpha * (X * X).sum(-1)
    base = [torch.zeros_like(alpha) for _ in range(L + 1)]
    for scale, omega in zip(*op):
        d2 = torch.ones_like(alpha) if omega == -1.0 else omega * omega / (omega * omega + alpha)
        for n, f in enumerate(_boys(L, T * d2)):
            base[n] = base[n] + scale * (-2.0 * alpha) ** n * d2 ** (n + 0.5) * f
    memo = {}

    def R(n, t):
        if (n, t) not in memo:
            if sum(t) == 0:
                return base[n]
            k = next(k for k in (0, 1, 2) if t[k])
            a = tuple(v - (1 if j == k else 0) for j, v in enumerate(t))
            v = X[..., k] * R(n + 1, a)
            if a[k]:
                v = v + a[k] * R(n + 1, tuple(w - (1 if j == k else 0) for j, w in enumerate(a)))
            memo[n, t] = v
        return memo[n, t]

    return {t: R(0, t) for t in _hermites(L)}


def _hermite_E(i, j, p, PA, PB):
    """E^{ij}_t, t = 0 .. i + j, of one axis."""
    e = [torch.ones_like(p)]
    for X in [PA] * i + [PB] * j:
        e = [(e[t - 1] / (2 * p) if t else 0) + (X * e[t] if t < len(e) else 0) + ((t + 1) * e[t + 1] if t + 1 < len(e) else 0)
             for t in range(len(e) + 1)]
    return e


class _Functions:
    """A basis as plain tensors; centres: (natom, 3), one point per atom."""

    def __init__(self, bas, centres=None, dev=None):
        P = bas.primitives
        self.dev = dev or torch.device("cuda" if torch.cuda.is_available() else "cpu")
        f = lambda v: torch.tensor(v, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.n, self.nao, self.pure = bas.ncart, bas.nao, bas.has_pure
        self.e, self.c = f([p.e for p in P]), f([p.c for p in P])
        self.L = np.array([p.L for p in P])
        self.cart = torch.tensor([p.cartIdx for p in P], device=self.dev)
        self.atom = torch.tensor([p.atomIdx for p in P], device=self.dev)
        self.xyz = f([[p.x, p.y, p.z] for p in P]) if centres is None else centres[self.atom]
        self.shells = sorted({(p.cartIdx, p.aoIdx, p.L, p.is_pure) for p in P})

    def to_cart(self):
        """nao x ncart: the real solid harmonics (m = 0, 1c, 1s, 2c, 2s for d)."""
        C = torch.zeros(self.nao, self.n, dtype=torch.float64, device=self.dev)
        r = math.sqrt(3.0)
        d = [[-0.5, 0, 0, -0.5, 0, 1.0], [0, 0, r, 0, 0, 0], [0, 0, 0, 0, r, 0], [r / 2, 0, 0, -r / 2, 0, 0],
             [0, r, 0, 0, 0, 0]]
        p = [[0, 0, 1.0], [1.0, 0, 0], [0, 1.0, 0]]
        for cart, ao, L, pure in self.shells:
            m = [[1.0]] if L == 0 else (d if L == 2 else p) if pure else np.eye((L + 1) * (L + 2) // 2).tolist()
            m = torch.tensor(m, dtype=torch.float64, device=self.dev)
            C[ao:ao + m.shape[0], cart:cart + m.shape[1]] = m
        return C


class _Pairs:
    """All primitive pairs of two bases by (L1, L2): exponents, centres, Hermite expansions
    (pair, Hermite, function pair) and the function pairs' indices a * n2 + b."""

    def __init__(self, f1, f2):
        self.blocks, self.shape = [], (f1.n, f2.n)
        for L1 in range(3):
            for L2 in range(3):
                i = torch.tensor(np.flatnonzero(f1.L == L1), device=f1.dev)
                j = torch.tensor(np.flatnonzero(f2.L == L2), device=f1.dev)
                i, j = i.repeat_interleave(len(j)), j.repeat(len(i))
                a, b, A, B = f1.e[i], f2.e[j], f1.xyz[i], f2.xyz[j]
                p = a + b
                K = f1.c[i] * f2.c[j] * torch.exp(-a * b / p * ((A - B) ** 2).sum(-1))
                keep = K.detach().abs() > 1.0e-18
                i, j, a, b, A, B, p, K = (v[keep] for v in (i, j, a, b, A, B, p, K))
                if not len(i):
                    continue
                P = (a[:, None] * A + b[:, None] * B) / p[:, None]
                E = [[[_hermite_E(m, n, p, P[:, k] - A[:, k], P[:, k] - B[:, k]) for n in range(L2 + 1)]
                      for m in range(L1 + 1)] for k in range(3)]
                cols = []
                for x, y in ((x, y) for x in _powers(L1) for y in _powers(L2)):
                    col = []
                    for t in _hermites(L1 + L2):
                        v = K
                        for k in range(3):
                            e = E[k][x[k]][y[k]]
                            v = v * e[t[k]] if t[k] < len(e) else None
                            if v is None:
                                break
                        col.append(torch.zeros_like(K) if v is None else v)
                    cols.append(torch.stack(col, 1))
                fa = f1.cart[i][:, None] + torch.arange(len(_powers(L1)), device=f1.dev)
                fb = f2.cart[j][:, None] + torch.arange(len(_powers(L2)), device=f1.dev)
                idx = (fa[:, :, None] * f2.n + fb[:, None, :]).reshape(len(i), -1)
                step = max(1, 60000 // len(_hermites(L1 + L2)))
                E = torch.stack(cols, 2)
                for o in range(0, len(i), step):
                    q = slice(o, o + step)
                    self.blocks.append((L1 + L2, p[q], P[q], E[q], idx[q], (L1, a[q], b[q], A[q], B[q], K[q])))


def _expand(block, nfun):
    """Hermite functions of a block x function pairs."""
    _, p, _, E, idx, _ = block
    n, H, F = E.shape
    M = torch.zeros(n, H, nfun, dtype=torch.float64, device=p.device)
    return M.scatter_add(2, idx[:, None, :].expand(n, H, F), E).reshape(n * H, nfun)


def _repulsion(bra, ket, op):
    """(ab|O|cd), function pairs x function pairs."""
    nb, nk = bra.shape[0] * bra.shape[1], ket.shape[0] * ket.shape[1]
    V = torch.zeros(nb, nk, dtype=torch.float64, device=bra.blocks[0][1].device)
    for y in ket.blocks:
        Wk = _expand(y, nk)
        Hk = _hermites(y[0])
        for x in bra.blocks:
            Hb = _hermites(x[0])
            step = max(1, 8000000 // len(y[1]))
            Wb = _expand(x, nb).reshape(len(x[1]), len(Hb), nb)
            for o in range(0, len(x[1]), step):
                p, P, q, Q = x[1][o:o + step, None], x[2][o:o + step, None, :], y[1][None], y[2][None]
                R = _hermite_R(x[0] + y[0], p * q / (p + q), P - Q, op)
                pref = 2.0 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q))
                R = torch.stack([torch.stack([pref * (-1) ** sum(u) * R[tuple(v + w for v, w in zip(t, u))] for u in Hk], 2)
                                 for t in Hb], 1)
                n = R.shape[0]
                V = V + Wb[o:o + step].reshape(n * len(Hb), nb).T @ (R.reshape(n * len(Hb), -1) @ Wk)
    return V.reshape(*bra.shape, *ket.shape)


def _back(f1, f2, M):
    return f1.to_cart() @ M @ f2.to_cart().T


def exact(case, seed):
    c = case
    if c["kind"] == "batch":
        return None
    inp = _inputs(c, seed)
    bas = inp[1]
    if c["kind"] == "one_electron":
        return _exact_one_electron(inp[0], bas) if bas.ncart <= 400 else None
    if max(bas.ncart, inp[2].ncart if c["kind"] == "fragments" else 0) > (30 if c["kind"] == "gradient" else 130):
        return None
    opJ, opK = _operators(c)
    if c["kind"] == "gradient":
        xyz = torch.tensor([[a.x, a.y, a.z] for a in inp[0].atoms], dtype=torch.float64,
                           device="cuda" if torch.cuda.is_available() else "cpu").requires_grad_()
        f = _Functions(bas, centres=xyz)
        D = f.to_cart().T @ torch.from_numpy(inp[2]).to(f.dev) @ f.to_cart()
        p = _Pairs(f, f)
        V = _repulsion(p, p, opJ)
        gJ, = torch.autograd.grad(torch.einsum("abcd,ab,cd", V, D, D), xyz, retain_graph=True)
        gK, = torch.autograd.grad(torch.einsum("abcd,ac,bd", V, D, D), xyz)
        return {"J": gJ.cpu().numpy(), "K": gK.cpu().numpy()}
    f = _Functions(bas)

    def both(fa, pj, pk, D):
        """J over the pairs of `pj` and K over those of `pk` on both sides, D in pure functions of fa."""
        C = fa.to_cart()
        D = C.T @ torch.from_numpy(D).to(fa.dev) @ C
        nb = pj[1].shape
        J = (_repulsion(pj[0], pj[1], opJ).reshape(-1, nb[0] * nb[1]) @ D.reshape(-1)).reshape(pj[0].shape)
        V = _repulsion(pk, pk, opK)
        n1, n2 = pk.shape
        # K_ac = sum_bd (ab|cd) D_bd
        K = V.permute(0, 2, 1, 3).reshape(n1 * n1, n2 * n2) @ D.reshape(-1)
        return J, K.reshape(n1, n1)

    if c["kind"] == "fragments":
        g = _Functions(inp[2])
        J, K = both(g, (_Pairs(f, f), _Pairs(g, g)), _Pairs(f, g), inp[3])
    else:
        p = _Pairs(f, f)
        J, K = both(f, (p, p), p, inp[2])
    if c["api"] == "host" or c["kind"] == "fragments":
        J, K = _back(f, f, J), _back(f, f, K)
    return {"J": J.cpu().numpy(), "K": K.cpu().numpy()}


def _exact_one_electron(mol, bas):
    f = _Functions(bas)
    Z = torch.tensor(np.asarray(mol.xyzZ), dtype=torch.float64, device=f.dev)
    n = f.n
    out = {k: torch.zeros(n * n, dtype=torch.float64, device=f.dev) for k in "STV"}
    for L, p, P, E, idx, (L1, a, b, A, B, K) in _Pairs(f, f).blocks:
        w = (math.pi / p) ** 1.5
        out["S"].index_add_(0, idx.reshape(-1), (E[:, 0, :] * w[:, None]).reshape(-1))
        # -1/2 d^2/dx^2 of a Gaussian of power j: -1/2 (j (j - 1) [j - 2] - 2 b (2 j + 1) [j] + 4 b^2 [j + 2])
        cols = []
        for x, y in ((x, y) for x in _powers(L1) for y in _powers(L - L1)):
            s = [[_hermite_E(x[k], max(m, 0), p, P[:, k] - A[:, k], P[:, k] - B[:, k])[0] if m >= 0 else 0
                  for m in (y[k] - 2, y[k], y[k] + 2)] for k in range(3)]
            t = [-0.5 * (y[k] * (y[k] - 1) * s[k][0] - 2 * b * (2 * y[k] + 1) * s[k][1] + 4 * b * b * s[k][2])
                 for k in range(3)]
            o = [v[1] for v in s]
            cols.append(K * w * (t[0] * o[1] * o[2] + o[0] * t[1] * o[2] + o[0] * o[1] * t[2]))
        out["T"].index_add_(0, idx.reshape(-1), torch.stack(cols, 1).reshape(-1))
        pot = []
        for o in range(0, len(p), 20000):
            q = slice(o, o + 20000)
            R = _hermite_R(L, p[q, None], P[q, None, :] - Z[None, :, :3], ([1.0], [-1.0]))
            pot.append(torch.stack([-(R[t] * Z[None, :, 3]).sum(1) * 2 * math.pi / p[q] for t in _hermites(L)], 1))
        v = (torch.cat(pot)[:, :, None] * E).sum(1)
        out["V"].index_add_(0, idx.reshape(-1), v.reshape(-1))
    return {k: _back(f, f, v.reshape(n, n)).cpu().numpy() for k, v in out.items()}
