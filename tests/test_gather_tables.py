"""The life of the gathers' index tables on the launch-recording build (tests/cpu_hip/recorder.py): their
cache is dropped when it outgrows its 64 MiB, and no launch may be given tables that were."""
import ctypes as C
import os
import sys
import threading

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_hip"))

from grassmanntn_amd import _lib as L  # noqa: E402
from grassmanntn_amd._perm import Perm  # noqa: E402
from recorder import recorder  # noqa: E402

BIG = 1 << 22  # entries of a table of 32 MiB, the largest
SRC, DST, STREAM = 1 << 40, 1 << 44, 0x3000


def _gather(n, big=BIG, enc=True):
    """A leg of `big` entries in the other encoder (one table) and one of n, exchanged; from a contiguous source."""
    P = Perm()
    i0, i1 = P.add_in(big, n, enc=enc), P.add_in(n, 1)
    v1 = P.add_virt(n)
    P.add_comp(v1, n, [(i1, 1)])
    P.add_out(n, [(v1, 1)])
    v0 = P.add_virt(big)
    P.add_comp(v0, big, [(i0, 1)])
    P.add_out(big, [(v0, 1)])
    return P.desc(L.GTN_F64, big * n)


def _permute(lib, d, stream=None):
    assert lib.gtn_permute(C.byref(d), C.c_void_p(SRC), C.c_void_p(DST), C.c_void_p(stream)) == 0


@pytest.fixture
def lib():
    r = recorder()
    r.rec_hold(None, b"", 0)
    r.rec_reset()
    yield r
    r.rec_hold(None, b"", 0)


def test_the_cache_is_dropped_and_rebuilt(lib):
    for n in (24, 40, 56, 24, 72):
        _permute(lib, _gather(n))
        assert lib.rec_live_bytes() < 130 << 20
    assert lib.rec_stale() == 0 and lib.rec_errors() == 0


def test_both_tables_of_a_double_gather(lib):
    """The second gather's table must not make room by dropping the first one's."""
    _permute(lib, _gather(88, big=1 << 10))
    for n in (48, 80, 96):
        inner = _gather(n)
        P = Perm()
        i0, i1 = P.add_in(n, BIG), P.add_in(BIG, 1, enc=True)
        for i, d in ((i1, BIG), (i0, n)):
            v = P.add_virt(d)
            P.add_comp(v, d, [(i, 1)])
            P.add_out(d, [(v, 1)])
        outer = P.desc(L.GTN_F64, BIG * n)
        assert lib.gtn_permute2(C.byref(outer), C.byref(inner), C.c_void_p(SRC), C.c_void_p(DST), None) == 0
    assert lib.rec_stale() == 0


def test_a_thread_about_to_launch_keeps_its_tables(lib):
    """A thread that has looked its tables up and stands before the launch; another outgrows the cache."""
    d = _gather(104)
    _permute(lib, d)
    lib.rec_hold(C.c_void_p(STREAM), b"k_permute", 0)
    a = threading.Thread(target=_permute, args=(lib, d, STREAM))
    a.start()
    b = threading.Thread(target=lambda: [_permute(lib, _gather(n)) for n in (112, 120, 136)])
    b.start()
    b.join(1)
    assert a.is_alive()
    lib.rec_hold(None, b"", 0)
    a.join(30)
    b.join(30)
    assert not a.is_alive() and not b.is_alive()
    assert lib.rec_stale() == 0


def test_tables_of_a_capture_are_kept(lib):
    """From the first capture to the last graph's end nothing that a graph may hold is dropped; that holds
    for the moments between the capture's end and the graph's making too."""
    alive, open_ = lib["_ZN3gtn12graphs_aliveEv"], lib["_ZN3gtn12capture_openEv"]
    seen = []
    hook = C.CFUNCTYPE(None)(lambda: seen.append(alive() or open_()))
    lib.rec_on_instantiate(hook)
    try:
        s, x = C.c_void_p(STREAM), C.c_void_p()
        assert lib.gtn_graph_begin(s, 1) == 0
        d = _gather(144)
        _permute(lib, d, STREAM)
        assert lib.gtn_graph_end(s, C.byref(x)) == 0
        for n in (152, 160, 168):
            _permute(lib, _gather(n))
        _permute(lib, d, STREAM)
        assert lib.rec_stale() == 0 and seen and all(seen)
        assert lib.gtn_graph_destroy(x) == 0
        assert not alive() and not open_()
    finally:
        lib.rec_on_instantiate(None)
