"""FP64 and FP32 grouped products at the edges of tiles and panels, in every operand layout, on aligned and
unaligned operands, against FP64 sums on the host."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")


# (M, N, K): around tiles of 64 and 128, panels of 8 and 16 (one, two, three and more of them), split reductions
@pytest.mark.parametrize("shape", [(1, 1, 1), (5, 3, 0), (64, 64, 8), (64, 64, 16), (64, 64, 24), (64, 64, 32), (65, 63, 7),
                                   (63, 65, 9), (128, 128, 40), (129, 127, 41), (200, 300, 25), (256, 130, 512),
                                   (64, 128, 1000), (32, 40, 4099)])
@pytest.mark.parametrize("layout", ["nn", "tn", "nt", "tt"])
@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("dtype,prec", [("f64", "f64"), ("f64", "f32"), ("f32", "f32"), ("f32", "f64")])
def test_products(shape, layout, pad, dtype, prec):
    """pad: elements before the operands and at the end of their rows (1: off 16-byte boundaries).  Rounding
    of the inputs (FP32), and of each of K sums, relative to the sum of absolute products."""
    from grassmanntn_amd import _lib as L
    from grassmanntn_amd._device import DeviceArray
    from grassmanntn_amd.core import _gemm, _gemm_desc
    m, n, k = shape
    rng = np.random.default_rng(m * 7 + n * 5 + k + pad)
    npd = np.float64 if dtype == "f64" else np.float32
    A, B = rng.standard_normal((2, m, k)).astype(npd), rng.standard_normal((2, k, n)).astype(npd)

    def hold(X, t):
        X = X.transpose(0, 2, 1) if t == "t" else X
        ld = X.shape[2] + pad
        out = np.full(pad + 2 * X.shape[1] * ld, np.nan, dtype=npd)  # what lies between must not be used
        v = out[pad:].reshape(2, X.shape[1], ld)
        v[:, :, :X.shape[2]] = X
        return DeviceArray.from_numpy(out), ld, X.shape[1] * ld

    dA, la, sab = hold(A, layout[0])
    dB, lb, sbb = hold(B, layout[1])
    C0 = rng.standard_normal((2, m, n)).astype(npd)
    dC = DeviceArray.from_numpy(C0)
    es = npd().itemsize
    sam, sak = (1, la) if layout[0] == "t" else (la, 1)
    sbk, sbn = (1, lb) if layout[1] == "t" else (lb, 1)
    for beta in (0.0, 0.5):
        d = _gemm_desc(dA.data_ptr() + es * pad, sam, sak, dB.data_ptr() + es * pad, sbk, sbn, dC.data_ptr(), n, 1, m, n, k,
                       batch=2, sab=sab, sbb=sbb, scb=m * n, alpha=-1.5, beta=beta)
        before = dC.numpy().astype(np.float64)
        _gemm([d], L.GTN_F64 if dtype == "f64" else L.GTN_F32, prec)
        a, b = A.astype(np.float64), B.astype(np.float64)
        if prec == "f32":
            a, b = a.astype(np.float32).astype(np.float64), b.astype(np.float32).astype(np.float64)
        want = -1.5 * (a @ b) + (beta * before if beta else 0.0)
        scale = 1.5 * np.abs(a) @ np.abs(b) + beta * np.abs(before)
        eps = 2.0 ** -24 if "f32" in (prec, dtype) else 2.0 ** -53
        got = dC.numpy().astype(np.float64)
        assert np.all(np.abs(got - want) <= eps * (k + 8) * scale + (2.0 ** -24 * np.abs(want) if dtype == "f32" else 0.0))
