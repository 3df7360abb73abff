"""How often the exchange gradient walks its pairs: once for densities that are symmetric, or symmetric
but for rounding (a spherical basis's d-d blocks, and any product of orbitals summed in another order,
differ from their transposes in the last bits), twice where both have an antisymmetric part.  The
launches of the call are counted in a process of its own; the results are compared as well: what
rounding leaves out is below 1e-25 of the largest elements' product.

    python tests/test_exchange_gradient_passes.py <built hipLaunchKernel> <basis>
"""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))

# hipLaunchKernel of the runtime, counting
SOURCE = r"""
#include <dlfcn.h>
#include <cstddef>
struct Dim3 { unsigned x, y, z; };
static long n = 0;
extern "C" long launches() { return n; }
extern "C" int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t lds, void* stream)
{
    using F = int (*)(const void*, Dim3, Dim3, void**, size_t, void*);
    static auto real = reinterpret_cast<F>(dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipLaunchKernel"));
    n++;
    return real(f, grid, block, args, lds, stream);
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "l.cpp").write_text(SOURCE)
    so = str(d / "l.so")
    subprocess.check_call(["g++", "-shared", "-fPIC", "-O1", str(d / "l.cpp"), "-o", so, "-ldl"])
    return so


@pytest.mark.parametrize("basis", ["cc-pvdz", "6-31gs"])
def test_passes(shim, basis):
    print("exchange gradient passes", basis, flush=True)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), shim, basis], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-4000:])


def main(so, basis):
    count = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)  # before liblsjk.so
    count.launches.restype = ctypes.c_long
    sys.path.insert(0, os.path.dirname(HERE))
    import lightspeed_amd as ls
    from lightspeed_amd import workloads as W
    bas = ls.Basis.from_gbs_file(W.water_cluster(1, 4.0, 1), basis)
    n = bas.nao
    rng = np.random.default_rng(1)
    A = rng.standard_normal((n, n))
    S = 0.5 * (A + A.T)
    noise = np.abs(S).max() * 2.0 ** -48 * rng.uniform(-1.0, 1.0, (n, n))
    anti = 1.0e-10 * (A - A.T)
    res, ew = ls.ResourceList.build(), ls.Ewald([1.0], [-1.0])
    pl = ls.PairList.build_schwarz(bas, bas, True, 1.0e-14)

    def grad(X, Y):
        x, y = (ls.Tensor.array(np.ascontiguousarray(v)) for v in (X, Y))
        before = count.launches()
        G = np.array(ls.IntBox.exchangeGrad(res, ew, pl, x, y, False, False, False, 1.0e-14, 1.0e-14).np)
        return G, count.launches() - before

    grad(S, S)
    G, once = grad(S, S)
    G1, l1 = grad(S + noise, S + noise.T)
    G2, l2 = grad(S + anti, S)
    G3, l3 = grad(S + anti, S + anti)
    G4, l4 = grad(A, A)
    classes = 36  # unordered pairs of s, p and d shells, six by six
    assert (once, l1, l2) == (l4 - classes,) * 3, (once, l1, l2, l3, l4)
    assert l3 == l4  # 1e-20 of the product, but there
    assert np.abs(G).max() > 0.1
    assert np.abs(G1 - G).max() < 1.0e-12 * np.abs(G).max()


if __name__ == "__main__":
    main(sys.argv[1], sys.argv[2])
