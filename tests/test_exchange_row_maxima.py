"""The exchange build without the sieve's row maxima (their scratch could not be allocated) against the
same build with them: the maxima only bound what a slot can reach, so the quartets are the same and K
differs by the order of its sums (1e-12).  A process of its own, in which the first allocation of the
first build is made to fail:

    python tests/test_exchange_row_maxima.py <built hipMalloc> <basis> <waters> <spread> <symm> <thredp>
"""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))

# hipMalloc of the runtime, but for the next allocation of an asked-for process (and its retries)
SOURCE = r"""
#include <dlfcn.h>
#include <cstddef>
static int next = 0;
static size_t failing = 0;
extern "C" void fail_next() { next = 1; }
extern "C" int hipMalloc(void** p, size_t n)
{
    static auto real = reinterpret_cast<int (*)(void**, size_t)>(dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipMalloc"));
    if (next) failing = n;
    next = 0;
    if (n == failing) return 2;  // hipErrorOutOfMemory
    failing = 0;
    return real(p, n);
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "m.cpp").write_text(SOURCE)
    so = str(d / "m.so")
    subprocess.check_call(["g++", "-shared", "-fPIC", "-O1", str(d / "m.cpp"), "-o", so, "-ldl"])
    return so


# one molecule's ket slots in part, all of them and none past the sieve; both routes
@pytest.mark.parametrize("basis,n,spread,symm,thredp", [
    ("6-31gs", 3, 1.0e-6, 1, 1.0e-12),
    ("6-31g", 6, 0.0, 0, 1.0e-12),
    ("cc-pvdz", 2, 1.0, 1, 1.0e-6),
])
def test_without_row_maxima(shim, basis, n, spread, symm, thredp):
    print("without row maxima", basis, n, spread, symm, thredp, flush=True)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), shim] + [str(v) for v in (basis, n, spread, symm, thredp)],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-4000:])


def main(so, basis, n, spread, symm, thredp):
    fail = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)  # before liblsjk.so
    sys.path.insert(0, os.path.dirname(HERE))
    import lightspeed_amd as ls
    from lightspeed_amd import workloads as W
    mol = W.water_cluster(n, W.water_cluster_box(n), 60 + n)
    bas = ls.Basis.from_gbs_file(mol, basis)
    frag = np.zeros(bas.ncart, int)
    for p in bas.primitives:
        frag[p.cartIdx:p.cartIdx + p.ncart] = p.atomIdx // 3
    A = np.random.default_rng(n).standard_normal((bas.ncart, bas.ncart))
    D = (A + A.T) * np.where(frag[:, None] == frag[None, :], 1.0, spread)
    pl = ls.PairList.build_schwarz(bas, bas, True, 1.0e-12)
    ls.IntBox.overlap(ls.ResourceList.build(), pl)  # the list's own arrays
    d, k = ls.DeviceArray(list(D.shape)), ls.DeviceArray(list(D.shape))
    d.upload(D)
    ls.set_counting(True)
    out = []
    for without in (True, False):
        k.upload(np.zeros_like(D))
        if without:
            fail.fail_next()  # the scratch is what the call allocates first
        ls.IntBox.exchange_device(ls.Ewald([1.0], [-1.0]), pl, pl, d.ptr, bool(symm), 1.0e-12, thredp, k.ptr)
        out.append((np.array(k.download()), np.array(ls.last_counts()), np.array(ls.last_counts_fp32())))
    (K1, c1, f1), (K2, c2, f2) = out
    assert np.abs(K2).max() > 0.1 and c2.sum() > 0
    assert np.array_equal(c1, c2)
    # (on the mixed route a wave step's precision depends on which slots share it)
    assert np.abs(K1 - K2).max() < (1.0e-12 if not f2.any() else 1.0e-7) * max(1.0, np.abs(K2).max())


if __name__ == "__main__":
    v = sys.argv
    main(v[1], v[2], int(v[3]), float(v[4]), int(v[5]), float(v[6]))
