"""The workspace of split reductions under several threads and streams, on the launch-recording build
(tests/cpu_hip/recorder.py): a use on another stream waits for the event behind the last use, within a
decomposition as well, and a thread in a decomposition does not keep others from their products."""
import ctypes as C
import os
import sys
import threading

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_hip"))

from grassmanntn_amd import _lib as L  # noqa: E402
from recorder import ops, recorder  # noqa: E402

S1, S2 = 0x1000, 0x2000


@pytest.fixture
def lib():
    r = recorder()
    r.gtn_autotune_set(0)
    r.rec_hold(None, b"", 0)
    r.rec_reset()
    yield r
    r.rec_hold(None, b"", 0)
    r.gtn_autotune_set(1)


def _decompose(lib, stream):
    """Two 1024 x 1024 blocks, 8 values each: split reductions all along."""
    b = (L.SvdBlock * 2)()
    for i in range(2):
        base = (i + 1) << 40
        b[i].M, b[i].U, b[i].S, b[i].Vt = base, base + (1 << 32), base + (2 << 32), base + (3 << 32)
        b[i].m = b[i].n = b[i].lda = b[i].ldv = 1024
        b[i].ldu = b[i].k = 8
    o = L.SvdOpts()
    o.oversample, o.iters, o.precision, o.seed, o.orth_every = 96, 20, 7, 1, 1
    n = lib.gtn_svd_workspace_bytes(b, 2, C.byref(o))
    assert lib.gtn_svd_blocks(b, 2, C.byref(o), C.c_void_p(1 << 45), C.c_int64(n), C.c_void_p(stream)) == 0


def _product(lib, stream):
    """64 x 64 x 8192: split into chunks."""
    d = L.GemmDesc()
    d.A, d.B, d.C = 1 << 41, 1 << 42, 1 << 43
    d.M, d.N, d.K, d.batch = 64, 64, 8192, 1
    d.sam, d.sak, d.sbk, d.sbn, d.scm, d.scn, d.alpha = 8192, 1, 64, 1, 64, 1, 1.0
    assert lib.gtn_gemm_grouped((L.GemmDesc * 1)(d), 1, L.GTN_F64, 0, C.c_void_p(stream)) == 0


def _uses(lib, log):
    """Indices of the reductions of split products."""
    return [i for i, o in enumerate(log) if o[0] == "L" and b"k_split_sum" in lib.rec_kernel(o[2])]


def _check_order(lib, log):
    """Between two uses on different streams, the first's stream records an event behind it, and the second's
    waits for that before it launches anything that could write there."""
    uses = _uses(lib, log)
    crossings = 0
    for a, b in zip(uses, uses[1:]):
        s, t = log[a][1], log[b][1]
        if s == t:
            continue
        crossings += 1
        wait = [i for i in range(a + 1, b) if log[i][0] == "W" and log[i][1] == t]
        assert wait, (a, b)
        rec = [i for i in range(a + 1, wait[-1]) if log[i][0] == "R" and log[i][1] == s and log[i][2] == log[wait[-1]][2]]
        assert rec, (a, b)
        writes = [i for i in range(wait[-1] + 1, b) if log[i][0] == "L" and log[i][1] == t]
        assert writes, (a, b)  # the partial products
    return crossings


def test_streams_one_after_another(lib):
    _product(lib, S1)
    _product(lib, S2)
    _decompose(lib, S1)
    _product(lib, S2)
    _product(lib, S2)
    _decompose(lib, S2)
    _decompose(lib, S1)
    log = ops(lib)
    assert _check_order(lib, log) == 4
    # one event for all reductions of a decomposition
    first = next(i for i, o in enumerate(log) if o[0] == "W" and o[1] == S1)
    last = next(i for i, o in enumerate(log) if i > first and o[0] == "W" and o[1] == S2)
    assert sum(1 for o in log[first:last] if o[0] == "R") == 1


@pytest.mark.parametrize("after", [0, 1, 2, 5, 18])
def test_products_pass_a_decomposition_of_another_thread(lib, after):
    """The decomposition's thread stands still after so many CholeskyQR rounds; a product on another stream (and
    one on the same) goes on, in order with the workspace's uses on both sides of it."""
    lib.rec_hold(C.c_void_p(S1), b"k_chol_inv", after)
    a = threading.Thread(target=_decompose, args=(lib, S1))
    a.start()
    try:
        while sum(1 for o in ops(lib) if o[0] == "L" and b"k_chol_inv" in lib.rec_kernel(o[2])) < after or not _uses(lib, ops(lib)):
            assert a.is_alive()
        b = threading.Thread(target=lambda: (_product(lib, S2), _product(lib, S2)))
        b.start()
        b.join(20)
        assert not b.is_alive() and a.is_alive()
    finally:
        lib.rec_hold(None, b"", 0)
        a.join(60)
        b.join(60)
    assert not a.is_alive()
    _product(lib, S2)
    assert _check_order(lib, ops(lib)) >= 1


@pytest.mark.gpu
def test_threads_on_their_own_streams():
    """A decomposition and a split product, each repeated by a thread on a stream of its own: bitwise what
    each gives alone (one workspace serves both)."""
    import numpy as np
    from grassmanntn_amd import core
    from grassmanntn_amd._device import DeviceArray
    dev = L.lib()
    rng = np.random.default_rng(1)
    m, k, K = 512, 8, 8192
    M = DeviceArray.from_numpy(rng.standard_normal((2, m, m)) * 0.98 ** np.arange(m))
    U, S, V = DeviceArray.zeros((2, m, k)), DeviceArray.zeros((2, k)), DeviceArray.zeros((2, k, m))
    b = (L.SvdBlock * 2)()
    for i in range(2):
        b[i].M, b[i].U = M.data_ptr() + 8 * i * m * m, U.data_ptr() + 8 * i * m * k
        b[i].S, b[i].Vt = S.data_ptr() + 8 * i * k, V.data_ptr() + 8 * i * k * m
        b[i].m = b[i].n = b[i].lda = b[i].ldv = m
        b[i].ldu = b[i].k = k
    o = L.SvdOpts()
    o.oversample, o.iters, o.precision, o.seed, o.orth_every = 96, 20, 7, 1, 1
    n = dev.gtn_svd_workspace_bytes(b, 2, C.byref(o))
    ws = DeviceArray.empty(n // 8)
    A, B = DeviceArray.from_numpy(rng.standard_normal((64, K))), DeviceArray.from_numpy(rng.standard_normal((K, 64)))
    P = DeviceArray.zeros((64, 64))
    d = (L.GemmDesc * 1)(core._gemm_desc(A.data_ptr(), K, 1, B.data_ptr(), 64, 1, P.data_ptr(), 64, 1, 64, 64, K))
    streams = [C.c_void_p(), C.c_void_p()]
    for s in streams:
        L.check(dev.gtn_stream_create(C.byref(s)), "stream")
    failures = []

    def decompose(reps, ref=None):
        for _ in range(reps):
            L.check(dev.gtn_svd_blocks(b, 2, C.byref(o), L.ptr(ws), n, streams[0]), "svd")
            L.check(dev.gtn_stream_synchronize(streams[0]), "wait")
            got = S.numpy()
            if ref is not None and not np.array_equal(got, ref):
                failures.append("values")
        return got

    def multiply(reps, ref=None):
        for _ in range(reps):
            L.check(dev.gtn_gemm_grouped(d, 1, L.GTN_F64, L.PREC["f64"], streams[1]), "gemm")
            L.check(dev.gtn_stream_synchronize(streams[1]), "wait")
            got = P.numpy()
            if ref is not None and not np.array_equal(got, ref):
                failures.append("product")
        return got

    L.check(dev.gtn_synchronize(), "sync")
    svd_ref, mul_ref = decompose(2), multiply(2)
    threads = [threading.Thread(target=decompose, args=(10, svd_ref)), threading.Thread(target=multiply, args=(200, mul_ref))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in streams:
        L.check(dev.gtn_stream_destroy(s), "stream")
    assert not failures, failures
