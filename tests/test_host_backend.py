"""The host side of liblsjk (layouts, buffers, launch decisions) on a machine without a GPU: hip_stub.cpp
stands in for the HIP runtime, "device" memory is host memory and kernels do not run.  Every case runs
in a process of its own, so that one that dies names itself:

    python tests/test_host_backend.py <built stub> <case>
"""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
THRE = 1.0e-12
CASES = {}


def case(f):
    CASES[f.__name__] = f
    return f


class Env:
    """The package over the stub."""

    def __init__(self, so):
        self.stub = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)  # before liblsjk.so
        for f in ("stub_uploaded", "stub_live_bytes"):
            getattr(self.stub, f).restype = ctypes.c_size_t
        for f in ("stub_bad_frees", "stub_null_stream_copies", "stub_live_blocks", "stub_launches", "stub_allocations",
                  "stub_event_waits"):
            getattr(self.stub, f).restype = ctypes.c_long
        self.stub.stub_launch_log.restype = ctypes.c_char_p
        self.stub.stub_launch_log.argtypes = [ctypes.c_long]
        self.stub.stub_unit.restype = ctypes.c_char_p
        self.stub.stub_unit.argtypes = [ctypes.c_long]
        self.stub.stub_fail_at.argtypes = [ctypes.c_long]
        self.stub.stub_answer.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
        sys.path[:0] = [ROOT, HERE]
        import capi_ctypes
        import lightspeed_amd as ls
        self.ls, self.C = ls, capi_ctypes
        self.res, self.ew = ls.ResourceList.build(), ls.Ewald([1.0], [-1.0])

    def basis(self, n, basis="6-31gs"):
        from lightspeed_amd import workloads as W
        return self.ls.Basis.from_gbs_file(W.water_cluster(n, W.water_cluster_box(n), n), basis)

    def pairs(self, b1, b2=None, thre=THRE):
        return self.ls.PairList.build_schwarz(b1, b2 or b1, b2 is None, thre)

    def tensor(self, *shape):
        return self.ls.Tensor.array(np.zeros(shape))

    def launches(self, part):
        return self.stub.stub_launches(part.encode())


@case
def copies_are_ordered(E):
    """No copy goes over the null stream, which does not order the library's streams, and none (nor a
    wait) falls into a graph's recording: lists made before, lists made by the call, results, counters."""
    I, t = E.ls.IntBox, THRE
    b1, b2 = E.basis(2), E.basis(1, "cc-pvdz")
    p1, p2 = E.pairs(b1), E.pairs(b2)
    E.ls.set_counting(True)
    for n, a, b in ((b1, p1, p1), (b2, p2, p2), (b2, p1, p2)):
        for thredp in (t, 1.0e-6):
            I.coulomb(E.res, E.ew, a, b, E.tensor(n.nao, n.nao), t, thredp)
    for symm in (True, False):
        I.exchange(E.res, E.ew, p1, p1, E.tensor(b1.nao, b1.nao), symm, t, 1.0e-6)
    E.ls.last_counts()
    E.ls.set_counting(False)
    D = E.tensor(b2.nao, b2.nao)
    I.coulombGrad(E.res, E.ew, p2, D, D, t, t)
    I.exchangeGrad(E.res, E.ew, p2, D, D, True, True, True, t, t)
    I.overlap(E.res, p2)
    I.potential(E.res, E.ew, p2, E.tensor(9, 4))
    d = E.ls.DeviceArray([b2.ncart, b2.ncart])
    E.ls.count_quartets(p2, p2, d.ptr, d.ptr, True, t)
    batch = E.ls.JKBatch.build(E.res, [p1, p2])
    buf = [E.ls.DeviceArray([batch.nelem]) for _ in range(3)]
    for thresp in (t, 1.0e-11, 1.0e-10, 1.0e-9, 1.0e-8, t):  # more thresholds than unit lists are kept for
        batch.jk_device(E.ew, buf[0].ptr, thresp, thresp, buf[1].ptr, buf[2].ptr)
    assert E.stub.stub_null_stream_copies() == 0


@case
def empty_lists(E):
    """Every entry point on a list without pairs adds nothing and returns."""
    I, t = E.ls.IntBox, THRE
    bas = E.basis(1)
    n = bas.nao
    none = E.pairs(bas, thre=1.0e10)
    some = E.pairs(bas)
    assert none.npair == 0 and some.npair > 0
    D = E.tensor(n, n)
    for a, b in ((none, none), (none, some), (some, none)):
        I.coulomb(E.res, E.ew, a, b, D, t, t)
        I.exchange(E.res, E.ew, a, b, D, True, t, t)
        I.exchange(E.res, E.ew, a, b, D, False, t, 1.0e-6)
    I.coulombGrad(E.res, E.ew, none, D, D, t, t)
    I.exchangeGrad(E.res, E.ew, none, D, D, True, True, True, t, t)
    I.overlap(E.res, none)
    I.kinetic(E.res, none)
    for charges in (0, 1, 300):
        I.potential(E.res, E.ew, none, E.tensor(charges, 4))
    d = E.ls.DeviceArray([n, n])
    E.ls.count_quartets(none, none, d.ptr, d.ptr, True, t)
    for lists in ([none], [none, some]):
        batch = E.ls.JKBatch.build(E.res, lists)
        buf = [E.ls.DeviceArray([batch.nelem]) for _ in range(3)]
        for _ in range(2):
            batch.jk_device(E.ew, buf[0].ptr, t, t, buf[1].ptr, buf[2].ptr)


@case
def call_buffers(E):
    """A block given back twice, or freed by lsjk_free, is refused and stays what it was; what is idle is
    bounded by 128 MiB and 16 blocks; a block given back busy is freed."""
    E.ls.hip_init(0)
    L = E.C.load()
    L.lsjk_buffer_acquire.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    L.lsjk_buffer_release.argtypes = [ctypes.c_void_p, ctypes.c_int]
    release = L.lsjk_buffer_release
    held_by_session = E.stub.stub_live_bytes(), E.stub.stub_live_blocks()

    def get(nbytes):
        p = ctypes.c_void_p()
        assert L.lsjk_buffer_acquire(ctypes.byref(p), nbytes) == 0
        return p.value

    def idle():
        """Bytes and blocks beyond the session's own (nothing is on loan)."""
        return E.stub.stub_live_bytes() - held_by_session[0], E.stub.stub_live_blocks() - held_by_session[1]

    mib = 1 << 20
    a = get(mib)
    assert L.lsjk_free(a) != 0  # on loan
    assert release(a, 0) == 0
    for busy in (0, 1):
        assert release(a, busy) != 0  # idle
    assert L.lsjk_free(a) != 0
    b, c = get(mib), get(mib)
    assert b == a and c != a  # not handed out twice
    assert release(b, 1) == 0 and release(c, 0) == 0
    assert idle() == (mib, 1)
    for p in [get(40 * mib) for _ in range(5)]:
        assert release(p, 0) == 0
    assert idle()[0] <= 128 * mib
    for p in [get(mib) for _ in range(40)]:
        assert release(p, 0) == 0
    nbytes, blocks = idle()
    assert blocks <= 16 and nbytes <= 128 * mib
    p = get(200 * mib)  # larger than all that may be idle
    assert release(p, 0) == 0 and idle() == (nbytes, blocks)
    p = get(3 * mib)
    assert idle()[1] == blocks + 1 and release(p, 1) == 0 and idle() == (nbytes, blocks)
    assert release(None, 0) == 0 and E.stub.stub_bad_frees() == 0
    assert L.lsjk_finalize() == 0 and E.stub.stub_bad_frees() == 0


@case
def exchange_without_row_maxima(E):
    """Where the scratch with the sieve's row maxima cannot be had, the build goes without them; so does a
    batch, whose graph is recorded all the same.  The next call is as ever."""
    bas = E.basis(3)
    n, t = bas.nao, THRE
    pl = E.pairs(bas)
    E.ls.IntBox.overlap(E.res, pl)  # the list's own arrays
    D, K = E.ls.DeviceArray([n, n]), E.ls.DeviceArray([n, n])

    def build(thredp):
        before = E.launches("k_rowmax"), E.launches("k_ket")
        E.ls.IntBox.exchange_device(E.ew, pl, pl, D.ptr, True, t, thredp, K.ptr)
        return E.launches("k_rowmax") - before[0], E.launches("k_ket") - before[1]

    E.stub.stub_fail_at(0)  # the call's scratch is what it allocates first
    rowmax, ket = build(t)
    assert rowmax == 0 and ket > 0
    assert build(t) == (1, ket)
    assert build(1.0e-6)[0] == 1

    def batch():
        b = E.ls.JKBatch.build(E.res, [pl, pl])
        return b, [E.ls.DeviceArray([b.nelem]) for _ in range(3)]

    def jk(b, buf, thredp=t):
        first = E.stub.stub_allocations(), E.launches("k_rowmax")
        b.jk_device(E.ew, buf[0].ptr, t, thredp, buf[1].ptr, buf[2].ptr)
        return E.stub.stub_allocations() - first[0], E.launches("k_rowmax") - first[1]

    jk(*batch())
    nalloc, rowmax = jk(*batch())
    assert rowmax == 2  # the call's own run and the recorded one
    b, buf = batch()
    E.stub.stub_fail_at(nalloc - 1)  # the graph's scratch is what it allocates last
    assert jk(b, buf) == (nalloc, 1)
    assert jk(b, buf) == (0, 0)  # replayed
    assert jk(b, buf, 1.0e-6)[1] == 1  # another graph, more scratch: again without
    E.ls.IntBox.coulomb_device(E.ew, pl, pl, D.ptr, t, t, K.ptr)


@case
def failed_allocations(E):
    """Whichever of its allocations a call fails at, the same call afterwards launches what it does on
    fresh lists."""
    I, t = E.ls.IntBox, THRE
    bas = E.basis(1, "6-31gs")
    D = E.tensor(bas.nao, bas.nao)
    calls = {
        "J": lambda p: I.coulomb(E.res, E.ew, p, p, D, t, t),
        "K": lambda p: I.exchange(E.res, E.ew, p, p, D, True, t, t),
        "K, general": lambda p: I.exchange(E.res, E.ew, p, p, D, False, t, t),
        "J gradient": lambda p: I.coulombGrad(E.res, E.ew, p, D, D, t, t),
        "K gradient": lambda p: I.exchangeGrad(E.res, E.ew, p, D, D, True, True, True, t, t),
        "V": lambda p: I.potential(E.res, E.ew, p, E.tensor(50, 4)),
    }

    def launches(f, p):
        first = E.launches("")
        f(p)
        return E.stub.stub_launch_log(first).decode()

    for name, f in calls.items():
        p = E.pairs(bas)
        n = E.stub.stub_allocations()
        fresh = launches(f, p)
        n = E.stub.stub_allocations() - n
        assert fresh and launches(f, p) == fresh
        failed = 0
        for k in range(n + 1):
            p = E.pairs(bas)
            E.stub.stub_fail_at(k)
            try:
                f(p)
            except RuntimeError:
                failed += 1
            E.stub.stub_fail_at(-1)
            assert launches(f, p) == fresh, (name, k)
        assert failed >= n // 2, (name, failed, n)


@case
def noalloc_scratch_limit(E):
    """lsjk_coulomb_noalloc takes what fits its 64 MiB (a float bound and H doubles per ket pair, H doubles
    per bra pair, each of the three rounded up to 256 bytes), here to the byte."""
    E.ls.hip_init(0)
    L, ptr = E.C.load(), ctypes.c_void_p
    n, m, H = 64000, 174760, 35  # pairs of two d functions
    r = lambda b: (b + 255) // 256 * 256  # noqa: E731
    assert r(4 * n) + r(8 * H * n) + r(8 * H * m) == 64 << 20

    def pairs(npair):
        nprim = int(np.ceil(np.sqrt(npair)))
        f, i = np.ones(nprim), np.arange(nprim, dtype=np.int32)
        xyz = np.linspace(0.0, 1.0, 3 * nprim)
        p = np.arange(npair)
        b, l = ptr(), ptr()
        two, cart = np.full(nprim, 2, np.int32), np.ascontiguousarray(6 * i)
        assert L.lsjk_basis_create(nprim, f.ctypes.data, f.ctypes.data, xyz.ctypes.data, two.ctypes.data, cart.ctypes.data,
                                   6 * nprim, ctypes.byref(b)) == 0
        p1, p2 = (np.ascontiguousarray(v, np.int32) for v in (p // nprim, p % nprim))
        bound = np.ones(npair, np.float32)
        assert L.lsjk_pairlist_create(b, b, 0, npair, p1.ctypes.data, p2.ctypes.data, bound.ctypes.data, ctypes.byref(l)) == 0
        return l

    bra, larger, ket = pairs(m), pairs(m + 1), pairs(n)
    D = np.zeros((6 * 253) ** 2)
    J = np.zeros((6 * 419) ** 2)
    one, bare = np.array([1.0]), np.array([-1.0])

    def call(f, bra, ket):
        return f(bra, ket, D.ctypes.data, 1, one.ctypes.data, bare.ctypes.data, THRE, THRE, J.ctypes.data)

    for b in (bra, larger):
        assert call(L.lsjk_coulomb, b, ket) == 0  # the task lists
    assert call(L.lsjk_coulomb_noalloc, bra, ket) == 0, L.lsjk_last_error()
    assert call(L.lsjk_coulomb_noalloc, larger, ket) != 0


@case
def first_pass_lists(E):
    """The first exchange over a list makes its scratch, six arrays per ket class and one unit list per
    launch, none for the mirror classes that do not run; the other route's first call makes no more."""
    bas = E.basis(2)
    pl = E.pairs(bas)
    E.ls.IntBox.overlap(E.res, pl)  # the list's own arrays
    D, K = E.ls.DeviceArray([bas.nao, bas.nao]), E.ls.DeviceArray([bas.nao, bas.nao])
    for thredp, expected in ((THRE, None), (1.0e-6, 0), (THRE, 0)):
        before = E.stub.stub_allocations(), E.launches("k_ket")
        E.ls.IntBox.exchange_device(E.ew, pl, pl, D.ptr, True, THRE, thredp, K.ptr)
        made, launched = E.stub.stub_allocations() - before[0], E.launches("k_ket") - before[1]
        assert launched == 45  # 81 classes of s, p and d rows and partners, 36 of them mirrors
        assert made == (1 + 6 * 9 + launched if expected is None else expected)


@case
def one_electron_streams(E):
    """Overlap, kinetic energy and the potential of few charges launch their classes in a row: fork and
    join of the side streams cost more than small classes gain by running side by side."""
    I = E.ls.IntBox
    pl = E.pairs(E.basis(3))

    def waits(f):
        f()
        before = E.stub.stub_event_waits()
        f()
        return E.stub.stub_event_waits() - before

    V = lambda n: waits(lambda: I.potential(E.res, E.ew, pl, E.tensor(n, 4)))  # noqa: E731
    assert waits(lambda: I.overlap(E.res, pl)) == waits(lambda: I.kinetic(E.res, pl)) == 0
    assert V(1) == V(9) == 0
    assert V(100000) > 0


@case
def exchange_code_by_operator(E):
    """The exchange kernels of one 1/r term and those of any terms are in code objects of their own, so that
    a process loads what it uses (k_ket's last template argument)."""
    kinds = []
    while E.stub.stub_unit(len(kinds)) is not None:
        names = [k for k in E.stub.stub_unit(len(kinds)).decode().split() if "5k_ketI" in k]
        kinds.append({k.split("5k_ketI")[1].split("EEEv")[0][-1] for k in names})
    assert sum(1 for k in kinds if k == {"1"}) == sum(1 for k in kinds if k == {"0"}) == 9
    assert all(len(k) <= 1 for k in kinds)


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.check_call(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", os.path.join(HERE, "hip_stub.cpp"), "-o", so])
    return so


@pytest.mark.parametrize("name", list(CASES))
def test_host(stub, name):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stub, name], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-4000:])


if __name__ == "__main__":
    CASES[sys.argv[2]](Env(sys.argv[1]))
