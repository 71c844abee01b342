"""gtn_mlp_mse with dout in the place of out, or of the only member's target: each element's gradient
replaces the value that it is made of, so the loss has to be summed first."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_hip"))


@pytest.mark.parametrize("where", ["apart", "out", "target", "half"])
def test_loss_is_summed_before_its_input_is_overwritten(where):
    """On the launch-recording build: a launch of the summing workgroups alone, then one of the writing ones."""
    from recorder import ops, recorder
    lib = recorder()
    E, n, c = (1 if where == "target" else 3), 5000, 17
    out, target, w, loss = 1 << 40, 1 << 41, 1 << 42, 1 << 43
    dout = {"apart": 1 << 44, "out": out, "target": target, "half": out + 2 * E * n * c}[where]
    lib.rec_reset()
    v = C.c_void_p
    assert lib.gtn_mlp_mse(v(out), v(target), v(w), C.c_int64(E), C.c_int64(n), C.c_int64(c), v(dout), v(loss), None) == 0
    launched = [o[3] for o in ops(lib) if o[0] == "L"]
    blocks = E * -(-n * c // 1024)
    assert launched == ([E + blocks] if where == "apart" else [E, blocks])


@pytest.mark.gpu
@pytest.mark.parametrize("E,n,c", [(1, 3, 17), (3, 4099, 17), (2, 300, 256)])
def test_in_place_equals_apart(E, n, c):
    from grassmanntn_amd import _lib as L
    from grassmanntn_amd._device import DeviceArray
    rng = np.random.default_rng(E + n + c)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    y, t, w = f(E, n, c), f(n, c), np.abs(f(c))
    dt, dw = DeviceArray.from_numpy(t), DeviceArray.from_numpy(w)

    def run(out, target, dout):
        loss = DeviceArray.zeros(E)
        L.check(L.lib().gtn_mlp_mse(L.ptr(out), L.ptr(target), L.ptr(dw), E, n, c, L.ptr(dout), L.ptr(loss), L.stream_ptr()),
                "mse")
        return dout.numpy(), loss.numpy()

    apart = run(DeviceArray.from_numpy(y), dt, DeviceArray.empty(y.shape, np.float32))
    d = DeviceArray.from_numpy(y)
    placed = run(d, dt, d)
    assert np.array_equal(placed[0], apart[0]) and np.array_equal(placed[1], apart[1])
    if E == 1:
        d = DeviceArray.from_numpy(t)
        placed = run(DeviceArray.from_numpy(y), d, d)
        assert np.array_equal(placed[0].reshape(apart[0].shape), apart[0]) and np.array_equal(placed[1], apart[1])
