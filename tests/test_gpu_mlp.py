"""GPU checks of the surrogate's kernels at the edges of their tiles and vectors, against FP64."""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")


def split(x, terms):
    """What the kernel multiplies: the sum of the leading BF16 terms of x."""
    out = np.zeros_like(x, dtype=np.float64)
    for _ in range(terms):
        out = out + M.bf16(x - out)
    return out


# (M, N, K): below, at and above a tile and a panel of the reduction, and reductions that are split
@pytest.mark.parametrize("shape", [(1, 1, 1), (64, 64, 32), (65, 63, 31), (128, 128, 64), (129, 200, 33), (100, 17, 256),
                                   (256, 17, 1030), (2, 256, 4096)])
@pytest.mark.parametrize("layout", ["nn", "tn", "nt", "tt"])
@pytest.mark.parametrize("dtype,prec,terms", [("f32", "bf16_split_a", (2, 1)), ("f32", "bf16", (1, 1)),
                                              ("f64", "bf16x3", (2, 2)), ("f64", "bf16x6", (3, 3))])
def test_bf16_products(shape, layout, dtype, prec, terms):
    """Products of split operands with exact terms: the error left is FP32 accumulation (2^-24 a term of the
    reduction, of the sum of absolute products) and, with two or three terms on both sides, the cross
    products left out (2^-16 and 2^-24 of it)."""
    from grassmanntn_amd import _lib as L
    from grassmanntn_amd._device import DeviceArray
    from grassmanntn_amd.core import _gemm, _gemm_desc
    m, n, k = shape
    rng = np.random.default_rng(m * 7 + n * 5 + k)
    npd = np.float32 if dtype == "f32" else np.float64
    A = rng.standard_normal((2, m, k)).astype(npd)
    B = rng.standard_normal((2, k, n)).astype(npd)
    hold = lambda X, t: np.ascontiguousarray(X.transpose(0, 2, 1) if t == "t" else X)  # noqa: E731
    dA, dB = DeviceArray.from_numpy(hold(A, layout[0])), DeviceArray.from_numpy(hold(B, layout[1]))
    dC = DeviceArray.zeros((2, m, n), npd)
    sam, sak = (1, m) if layout[0] == "t" else (k, 1)
    sbk, sbn = (1, k) if layout[1] == "t" else (n, 1)
    d = _gemm_desc(dA.data_ptr(), sam, sak, dB.data_ptr(), sbk, sbn, dC.data_ptr(), n, 1, m, n, k, batch=2, sab=m * k,
                   sbb=k * n, scb=m * n)
    _gemm([d], L.GTN_F32 if dtype == "f32" else L.GTN_F64, prec)
    sa, sb = split(A.astype(np.float64), terms[0]), split(B.astype(np.float64), terms[1])
    scale = np.abs(sa) @ np.abs(sb)
    left_out = 0.0 if terms[1] == 1 else 4 * 2.0 ** (-8 * terms[0])
    assert np.all(np.abs(dC.numpy() - sa @ sb) <= (2.0 ** -23 * (k + 4) + left_out) * scale)


@pytest.mark.parametrize("E,n,c", [(1, 1, 1), (2, 3, 17), (5, 100, 64), (3, 77, 200), (2, 4099, 256), (2, 1025, 6)])
def test_elementwise_stages(E, n, c):
    """Bias, GELU, its derivative and the loss over odd and vector-sized rows: FP32 rounding of each result."""
    from grassmanntn_amd import _lib as L
    from grassmanntn_amd._device import DeviceArray
    rng = np.random.default_rng(E + n + c)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    y, b, t, w = f(E, n, c), f(E, c), f(n, c), np.abs(f(c))
    dy, db, dt, dw = (DeviceArray.from_numpy(x) for x in (y, b, t, w))
    pre, dout, loss = DeviceArray.empty(y.shape, np.float32), DeviceArray.empty(y.shape, np.float32), DeviceArray.zeros(E)
    lib, s = L.lib(), L.stream_ptr()
    L.check(lib.gtn_mlp_mse(L.ptr(dy), L.ptr(dt), L.ptr(dw), E, n, c, L.ptr(dout), L.ptr(loss), s), "mse")
    L.check(lib.gtn_mlp_bias_act(L.ptr(dy), E, n, c, L.ptr(db), L.GTN_ACT_GELU, L.ptr(pre), s), "bias_act")
    L.check(lib.gtn_mlp_act_backward(L.ptr(dout), L.ptr(pre), E * n * c, L.GTN_ACT_GELU, s), "act_backward")
    d = y.astype(np.float64) - t
    np.testing.assert_allclose(loss.numpy(), (w * d * d).sum(axis=(1, 2)) / n, rtol=1e-12)
    p = (y + b[:, None, :]).astype(np.float32)
    assert np.array_equal(pre.numpy(), p)
    p = p.astype(np.float64)
    np.testing.assert_allclose(dy.numpy(), M.gelu(p), rtol=0, atol=4e-7 * (1 + np.abs(p).max()))
    g = 2 * w * d / n
    np.testing.assert_allclose(dout.numpy(), g * M.gelu_grad(p), rtol=0, atol=4e-7 * (1 + np.abs(p).max()) * np.abs(g).max())
