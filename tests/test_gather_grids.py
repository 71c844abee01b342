"""The grids that gtn_permute launches for gathers of many elements, on the launch-recording build of its
sources (tests/cpu_hip/recorder.py): no kernel runs and nothing of the tensors' size is allocated.  HIP
refuses a dimension of 2^32 work items and more."""
import ctypes as C
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_hip"))

from grassmanntn_amd import _lib as L  # noqa: E402
from grassmanntn_amd._perm import Perm, strides  # noqa: E402
from recorder import ops, recorder  # noqa: E402


def _transpose(shape, order):
    """out axis a = source axis order[a] of a contiguous tensor of plain (bosonic) legs."""
    P = Perm()
    st = strides(shape)
    ins = [P.add_in(n, s) for n, s in zip(shape, st)]
    for b in order:
        v = P.add_virt(shape[b])
        P.add_comp(v, shape[b], [(ins[b], 1)])
        P.add_out(shape[b], [(v, 1)])
    return P


# tiles of 16 x 16 (2^32 elements), pairs of extents just above 16 (four mostly empty tiles a pair), 64 x 64
# tiles, rows of 256 and of 1024 columns, and an element walk
@pytest.mark.parametrize("shape,order", [((16, 1 << 12, 1 << 12, 16), (3, 1, 2, 0)), ((16, 1 << 24, 16), (2, 1, 0)),
                                         ((17, 2048, 2050, 17), (3, 1, 2, 0)), ((17, 1 << 22, 17), (2, 1, 0)),
                                         ((16, 1 << 25, 16), (2, 1, 0)), ((64, 1 << 21, 64), (2, 1, 0)),
                                         ((1 << 14, 1 << 13, 256), (1, 0, 2)), ((1 << 13, 1 << 14, 768), (1, 0, 2)),
                                         ((1 << 15, 1 << 14, 7), (1, 0, 2)), ((16, 1 << 20, 16), (2, 1, 0))])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_gathers_of_many_elements_launch(shape, order, dtype):
    lib = recorder()
    n = 1
    for d in shape:
        n *= d
    d = _transpose(shape, order).desc(L.GTN_F64 if dtype == "f64" else L.GTN_F32, n)
    lib.rec_reset()
    rc = lib.gtn_permute(C.byref(d), C.c_void_p(1 << 40), C.c_void_p(1 << 44), None)
    launched = [o for o in ops(lib) if o[0] == "L"]
    assert rc == 0 and lib.rec_errors() == 0
    assert launched and all(o[3] * o[4] < 1 << 32 for o in launched)
