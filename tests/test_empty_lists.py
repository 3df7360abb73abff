"""Lists without pairs (two bases out of each other's reach, a threshold above every bound) through
every entry point: results are exactly zero, alone and beside a list that has pairs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

THRE = 1.0e-12


@pytest.mark.parametrize("apart", [False, True])
def test_empty_lists(product_backend, apart):
    ls = product_backend.ls
    from lightspeed_amd import workloads as W
    print("empty lists", apart, flush=True)
    mol = W.water_cluster(1, 4.0, 1)
    bas = ls.Basis.from_gbs_file(mol, "6-31gs")
    res, ew, I = ls.ResourceList.build(), ls.Ewald([0.5, 0.5], [-1.0, 0.3]), ls.IntBox
    D = ls.Tensor.array(np.random.default_rng(1).standard_normal((bas.nao, bas.nao)))
    some = ls.PairList.build_schwarz(bas, bas, True, THRE)
    if apart:
        far = ls.Basis.from_gbs_file(ls.Molecule("far", [a._replace(x=a.x + 500.0) for a in mol.atoms]), "6-31gs")
        none = ls.PairList.build_schwarz(bas, far, False, THRE)
    else:
        none = ls.PairList.build_schwarz(bas, bas, True, 1.0e10)
    assert none.npair == 0 and some.npair > 0
    out = [I.overlap(res, none), I.kinetic(res, none)]
    for n in (1, 300):
        out.append(I.potential(res, ew, none, ls.Tensor.array(np.ones((n, 4)))))
    for a, b in ((none, none), (none, some), (some, none)):
        for thredp in (THRE, 1.0e-6):
            out.append(I.coulomb(res, ew, a, b, D, THRE, thredp))
            out.append(I.exchange(res, ew, a, b, D, a is b, THRE, thredp))
    if not apart:
        out.append(I.coulombGrad(res, ew, none, D, D, THRE, THRE))
        out.append(I.exchangeGrad(res, ew, none, D, D, True, True, True, THRE, THRE))
    for M in out:
        assert not np.array(M.np).any()
