"""The branches of the builds that the fixtures do not reach at their edges, each against the oracle at
the same screening thresholds (so the same quartets: differences are FP64 rounding, 1e-10 as in the
parity tests)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1.0e-10
MULTI = ([0.7, -0.4, 1.2], [-1.0, 0.3, 2.0])  # 1/r and two erf terms


def _waters(ls, basis, n):
    from lightspeed_amd import workloads as W
    mol = W.water_cluster(n, W.water_cluster_box(n), 60 + n)
    return mol, ls.Basis.from_gbs_file(mol, basis)


def _fragment_density(bas, rng, symm, spread):
    """Blocks within each molecule, the others scaled by `spread`; one molecule's rows exactly zero."""
    frag = np.zeros(bas.nao, int)
    for p in bas.primitives:
        frag[p.aoIdx:p.aoIdx + (2 * p.L + 1 if p.is_pure else p.ncart)] = p.atomIdx // 3
    D = rng.standard_normal((bas.nao, bas.nao)) * np.where(frag[:, None] == frag[None, :], 1.0, spread)
    if frag.max() > 0:
        D[frag == 0, :] = 0.0
    return np.ascontiguousarray(0.5 * (D + D.T) if symm else D)


# the sieve of K's ket slots: lists below one wave's slots and above it, all slots failing, few or most
# passing, directly walked and gathered D blocks, one term (the 1/r kernels) and several
@pytest.mark.parametrize("basis,n,symm,spread,op", [
    ("sto-3g", 1, True, 1.0, ([1.0], [-1.0])),
    ("6-31g", 6, True, 0.0, ([1.0], [-1.0])),
    ("6-31g", 6, False, 1.0e-9, ([1.0], [-1.0])),
    ("6-31g", 4, True, 1.0e-7, MULTI),
    ("cc-pvdz", 2, False, 1.0e-9, ([1.0], [-1.0])),
])
def test_exchange_sieve(product_backend, oracle_backend, basis, n, symm, spread, op):
    ls, O = product_backend.ls, oracle_backend.O
    print("exchange sieve", basis, n, symm, spread, flush=True)
    mol, bas = _waters(ls, basis, n)
    D = _fragment_density(bas, np.random.default_rng(n), symm, spread)
    pl = ls.PairList.build_schwarz(bas, bas, True, 1.0e-12)
    ob = O.OBasis(bas)
    opl = O.OPairList(ob, ob, True, 1.0e-12)
    counts = np.zeros(625, np.int64)
    Ko = O.exchange(op, opl, opl, D, False, 1.0e-12, counts=counts)
    res, ew = ls.ResourceList.build(), ls.Ewald(*op)
    ls.set_counting(True)
    try:
        K = ls.IntBox.exchange(res, ew, pl, pl, ls.Tensor.array(D), False, 1.0e-12, 1.0e-12).np
        kc = ls.last_counts()
    finally:
        ls.set_counting(False)
    assert np.abs(K - Ko).max() < TOL
    # the oracle counts a quartet once per operator term, the kernels once
    assert np.array_equal(kc[256:256 + 625].astype(np.int64) * len(op[0]), counts)
    if symm:
        K = ls.IntBox.exchange(res, ew, pl, pl, ls.Tensor.array(D), True, 1.0e-12, 1.0e-12).np
        assert np.abs(K - O.exchange(op, opl, opl, D, True, 1.0e-12)).max() < TOL


# J from Boys functions (orders 2 to 4) under several terms and under one, over one list and over two
@pytest.mark.parametrize("op", [MULTI, ([1.0], [0.4]), ([-1.0], [-1.0])])
@pytest.mark.parametrize("two", [False, True])
def test_coulomb_operators(product_backend, oracle_backend, op, two):
    ls, O = product_backend.ls, oracle_backend.O
    print("coulomb operators", op, two, flush=True)
    mol, bas = _waters(ls, "cc-pvdz", 2)
    other = _waters(ls, "6-31gs", 3)[1] if two else bas
    rng = np.random.default_rng(5)
    D = rng.standard_normal((other.nao, other.nao))
    D = np.ascontiguousarray(0.5 * (D + D.T))
    p12 = ls.PairList.build_schwarz(bas, bas, True, 1.0e-12)
    p34 = ls.PairList.build_schwarz(other, other, True, 1.0e-12) if two else p12
    o1, o2 = O.OBasis(bas), O.OBasis(other)
    q12 = O.OPairList(o1, o1, True, 1.0e-12)
    q34 = O.OPairList(o2, o2, True, 1.0e-12) if two else q12
    J = ls.IntBox.coulomb(ls.ResourceList.build(), ls.Ewald(*op), p12, p34, ls.Tensor.array(D), 1.0e-12, 1.0e-12).np
    assert np.abs(J - O.coulomb(op, q12, q34, D, 1.0e-12)).max() < TOL


# the potential's charges in one part and cut into several, the last part shorter
@pytest.mark.parametrize("basis,n,ncharge", [("sto-3g", 1, 1), ("cc-pvdz", 1, 17), ("6-31gs", 3, 301)])
@pytest.mark.parametrize("op", [MULTI, ([1.0], [-1.0])])
def test_potential_charges(product_backend, oracle_backend, basis, n, ncharge, op):
    ls, O = product_backend.ls, oracle_backend.O
    print("potential", basis, n, ncharge, flush=True)
    mol, bas = _waters(ls, basis, n)
    rng = np.random.default_rng(ncharge)
    xyzc = np.ascontiguousarray(np.concatenate([rng.uniform(-6, 6, (ncharge, 3)), rng.uniform(-1, 1, (ncharge, 1))], 1))
    xyzc[0, :3] = [mol.atoms[0].x, mol.atoms[0].y, mol.atoms[0].z]  # one on a nucleus
    pl = ls.PairList.build_schwarz(bas, bas, True, 1.0e-14)
    ob = O.OBasis(bas)
    V = ls.IntBox.potential(ls.ResourceList.build(), ls.Ewald(*op), pl, ls.Tensor.array(xyzc)).np
    assert np.abs(V - O.potential(op, O.OPairList(ob, ob, True, 1.0e-14), xyzc)).max() < TOL


def test_coulomb_gradient_of_one_density(product_backend):
    """One tensor in both roles (one half, doubled) against two tensors of the same values."""
    ls = product_backend.ls
    mol, bas = _waters(ls, "6-31gs", 2)
    A = np.random.default_rng(2).standard_normal((bas.nao, bas.nao))
    D = np.ascontiguousarray(0.5 * (A + A.T))
    pl = ls.PairList.build_schwarz(bas, bas, True, 1.0e-12)
    res, ew, t = ls.ResourceList.build(), ls.Ewald([1.0], [-1.0]), ls.Tensor.array(D)
    one = ls.IntBox.coulombGrad(res, ew, pl, t, t, 1.0e-14, 1.0e-14).np
    two = ls.IntBox.coulombGrad(res, ew, pl, t, ls.Tensor.array(D.copy()), 1.0e-14, 1.0e-14).np
    # both leave out quartets below 1e-14 (fewer than 1e6 of them), each half by its own bounds
    assert np.abs(one - two).max() < 1.0e-8 * max(1.0, np.abs(two).max())


def test_call_buffers(product_backend):
    """A released block serves the next request of its size, one that may be in use does not stay, and
    the idle ones are bounded; builds of alternating sizes give what they gave."""
    import capi_ctypes
    ls = product_backend.ls
    res, ew = ls.ResourceList.build(), ls.Ewald([1.0], [-1.0])
    ref = {}
    for _ in range(2):
        for n in (1, 5, 2):
            mol, bas = _waters(ls, "6-31g", n)
            D = np.eye(bas.nao)
            pl = ls.PairList.build_schwarz(bas, bas, True, 1.0e-12)
            J = np.array(ls.IntBox.coulomb(res, ew, pl, pl, ls.Tensor.array(D), 1.0e-12, 1.0e-12).np)
            assert np.abs(J - ref.setdefault(n, J)).max() < 1.0e-11
            with pytest.raises(Exception):
                ls.IntBox.coulomb(res, ew, pl, pl, ls.Tensor.array(np.eye(bas.nao + 1)), 1.0e-12, 1.0e-12)
    L = capi_ctypes.load()
    acquire, release = L.lsjk_buffer_acquire, L.lsjk_buffer_release
    acquire.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    release.argtypes = [ctypes.c_void_p, ctypes.c_int]

    def get(nbytes):
        p = ctypes.c_void_p()
        assert acquire(ctypes.byref(p), nbytes) == 0
        return p.value

    mib = 1 << 20
    a = get(9 * mib)
    assert release(a, 0) == 0
    b = get(9 * mib - 5)  # the same block
    c = get(9 * mib)      # that one is on loan
    assert b == a and c != a
    assert release(b, 1) == 0 and release(c, 0) == 0
    held = [get(40 * mib) for _ in range(5)]  # more than stays
    assert len(set(held)) == 5
    for p in held:
        assert release(p, 0) == 0
    again = [get(40 * mib) for _ in range(5)]
    assert len(set(again) & set(held)) >= 1
    for p in again:
        assert release(p, 1) == 0
    assert acquire(None, 8) != 0
