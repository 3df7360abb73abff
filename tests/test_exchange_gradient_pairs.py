"""Exchange gradient against an FP64 reference without screening (perf/cases.py: Hermite expansion of
all function pairs, derivatives by automatic differentiation), over what the pair-of-pairs kernel
distinguishes: every class up to (dd|dd), lists shorter and longer than one tile of 64 pairs, erf
operators, and densities with antisymmetric parts (both, one, none; the same or two matrices).

Tolerance: quartets below thresp = 1e-14 are left out, about 1e6 of them at the largest size with
random signs (1e-11), and FP64 rounding of sums of order 10 (1e-14 each term): 1e-9, as the fixtures.
"""
import importlib.util
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _reference():
    spec = importlib.util.spec_from_file_location("perf_cases_reference", os.path.join(ROOT, "perf", "cases.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


@pytest.mark.parametrize("basis,n,op,kind", [
    ("sto-3g", 1, ([1.0], [-1.0]), "same"),
    ("6-31gs", 1, ([1.0], [-1.0]), "two_general"),
    ("6-31gs", 1, ([0.3, -0.7], [-1.0, 0.4]), "general"),
    ("cc-pvdz", 1, ([1.0], [0.5]), "one_general"),
    ("sto-3g", 3, ([1.0], [-1.0]), "two_general"),
])
def test_against_unscreened_reference(basis, n, op, kind):
    M = _reference()
    import torch
    ls = M.ls
    mol = M.W.water_cluster(n, M.W.water_cluster_box(n), 40 + n)
    bas = ls.Basis.from_gbs_file(mol, basis)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((bas.nao, bas.nao)) * 0.3
    Y = rng.standard_normal((bas.nao, bas.nao)) * 0.3
    sym = lambda A: 0.5 * (A + A.T)  # noqa: E731
    D13, D24 = {"same": (sym(X), sym(X)), "general": (X, X), "two_general": (X, Y), "one_general": (X, sym(Y))}[kind]
    print("exchange gradient", basis, n, kind, "nao", bas.nao, flush=True)
    xyz = torch.tensor([[a.x, a.y, a.z] for a in mol.atoms], dtype=torch.float64).requires_grad_()
    f = M._Functions(bas, centres=xyz, dev=xyz.device)
    p = M._Pairs(f, f)
    V = M._repulsion(p, p, op)
    C = f.to_cart()
    A, B = (C.T @ torch.from_numpy(np.ascontiguousarray(d)) @ C for d in (D13, D24))
    ref, = torch.autograd.grad((V.permute(0, 2, 1, 3) * A[:, :, None, None] * B).sum(), xyz)
    ref = ref.numpy()
    pl = ls.PairList.build_schwarz(bas, bas, True, 1.0e-14)
    res = ls.ResourceList.build()
    ta = ls.Tensor.array(np.ascontiguousarray(D13))
    tb = ta if kind == "same" else ls.Tensor.array(np.ascontiguousarray(D24))
    s13, s24 = kind == "same", kind in ("same", "one_general")
    G = ls.IntBox.exchangeGrad(res, ls.Ewald(*op), pl, ta, tb, s13, s24, kind == "same", 1.0e-14, 1.0e-14).np
    err = np.abs(np.array(G) - ref).max()
    print("  max|dG| %.1e of %.1e" % (err, np.abs(ref).max()), flush=True)
    assert np.abs(ref).max() > 0.01 and err < 1.0e-9
