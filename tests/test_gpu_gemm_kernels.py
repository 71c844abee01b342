"""Each kernel of the grouped products in each of its launch configurations, whatever the autotuner would
choose: the plain and the pipelined kernel, 64 and 128 wide tiles, with and without a split reduction, on
panels that end whole and not, aligned and unaligned rows, and symmetric products' one triangle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")

KINDS = [("f64", "f64"), ("f32", "f32"), ("f32", "f64"), ("f64", "f32")]


def _launch(d, dtype, prec, tile, target, kernel, symmetric=0):
    from grassmanntn_amd import _lib as L
    arr = (L.GemmDesc * len(d))(*d)
    L.check(L.lib().gtn_gemm_grouped_as(arr, len(d), L.GTN_F64 if dtype == "f64" else L.GTN_F32, L.PREC[prec], tile, target,
                                        kernel, symmetric, L.stream_ptr()), "gtn_gemm_grouped_as")


# (M, N, K): one, two, three and more panels of 8 and 16, remainders, edge tiles, chunks of a split reduction
SHAPES = [(1, 1, 1), (64, 64, 8), (64, 64, 16), (65, 63, 7), (64, 128, 25), (128, 128, 24), (128, 128, 32), (128, 130, 40),
          (129, 191, 41), (192, 256, 64), (130, 128, 1031), (256, 128, 2048)]


@pytest.mark.parametrize("dtype,prec", KINDS)
@pytest.mark.parametrize("kernel,tile,target", [(k, t, s) for k in (0, 1) for t in (64, 128) for s in (0, 1024)])
def test_every_configuration(dtype, prec, kernel, tile, target):
    """Errors: the rounding of each of K sums (and of the inputs, in FP32) of the sum of absolute products."""
    from grassmanntn_amd._device import DeviceArray
    from grassmanntn_amd.core import _gemm_desc
    if kernel and (dtype, prec) == ("f64", "f32"):
        pytest.skip("FP32 arithmetic on FP64 operands has one kernel")
    npd = np.float64 if dtype == "f64" else np.float32
    es = npd().itemsize
    for m, n, k in SHAPES:
        if tile == 128 and min(m, n) < 128:
            continue
        for layout in ("nn", "tn", "nt", "tt"):
            for pad in (0, 1):
                rng = np.random.default_rng(m + n + k + pad)
                A, B = rng.standard_normal((2, m, k)).astype(npd), rng.standard_normal((2, k, n)).astype(npd)

                def hold(X, t):
                    X = X.transpose(0, 2, 1) if t == "t" else X
                    ld = X.shape[2] + pad
                    out = np.full(pad + 2 * X.shape[1] * ld, np.nan, dtype=npd)  # what lies between must not be used
                    out[pad:].reshape(2, X.shape[1], ld)[:, :, :X.shape[2]] = X
                    return DeviceArray.from_numpy(out), ld, X.shape[1] * ld

                dA, la, sab = hold(A, layout[0])
                dB, lb, sbb = hold(B, layout[1])
                C0 = rng.standard_normal((2, m, n)).astype(npd)
                dC = DeviceArray.from_numpy(C0)
                sam, sak = (1, la) if layout[0] == "t" else (la, 1)
                sbk, sbn = (1, lb) if layout[1] == "t" else (lb, 1)
                d = _gemm_desc(dA.data_ptr() + es * pad, sam, sak, dB.data_ptr() + es * pad, sbk, sbn, dC.data_ptr(), n, 1, m, n,
                               k, batch=2, sab=sab, sbb=sbb, scb=m * n, alpha=-1.5, beta=0.5)
                _launch([d], dtype, prec, tile, target, kernel)
                a, b = A.astype(np.float64), B.astype(np.float64)
                if prec == "f32":
                    a, b = a.astype(np.float32).astype(np.float64), b.astype(np.float32).astype(np.float64)
                want = -1.5 * (a @ b) + 0.5 * C0
                scale = 1.5 * np.abs(a) @ np.abs(b) + 0.5 * np.abs(C0)
                eps = 2.0 ** -24 if "f32" in (prec, dtype) else 2.0 ** -53
                assert np.all(np.abs(dC.numpy() - want) <= eps * (k + 8) * scale), (m, n, k, layout, pad)


@pytest.mark.parametrize("kernel,tile,target", [(k, t, s) for k in (0, 1) for t in (64, 128) for s in (0, 512, 1024)])
def test_symmetric_products(kernel, tile, target):
    """Two groups, two blocks each: M M^T from its upper tiles, the same on both sides to the bit."""
    from grassmanntn_amd._device import DeviceArray
    from grassmanntn_amd.core import _gemm_desc
    for sizes in (((128, 40), (191, 64)), ((193, 2048), (256, 7)), ((320, 129), (129, 1030))):
        d, held = [], []
        for m, k in sizes:
            M = np.random.default_rng(m + k).standard_normal((2, m, k))
            dM, dG = DeviceArray.from_numpy(M), DeviceArray.from_numpy(np.full((2, m, m), np.nan))
            d.append(_gemm_desc(dM.data_ptr(), k, 1, dM.data_ptr(), 1, k, dG.data_ptr(), m, 1, m, m, k, batch=2, sab=m * k,
                                sbb=m * k, scb=m * m))
            held.append((M, dM, dG))
        _launch(d, "f64", "f64", tile, target, kernel, symmetric=1)
        for M, _dM, dG in held:
            G = dG.numpy()
            assert np.array_equal(G, G.transpose(0, 2, 1))
            bound = 2.0 ** -53 * (M.shape[2] + 8) * (np.abs(M) @ np.abs(M.transpose(0, 2, 1)))
            assert np.all(np.abs(G - M @ M.transpose(0, 2, 1)) <= bound)


def test_configurations_out_of_range_are_refused():
    from grassmanntn_amd import _lib as L
    from grassmanntn_amd._device import DeviceArray
    from grassmanntn_amd.core import _gemm_desc
    x = DeviceArray.zeros((64, 64))
    d = _gemm_desc(x.data_ptr(), 64, 1, x.data_ptr(), 64, 1, x.data_ptr(), 64, 1, 64, 64, 64)
    for bad in (("f64", "f64", 128, 0, 0), ("f64", "f64", 32, 0, 0), ("f64", "f64", 64, -1, 0), ("f64", "f64", 64, 0, 2),
                ("f64", "f32", 64, 0, 1), ("f64", "bf16", 64, 0, 1)):
        with pytest.raises(L.GrassmannDeviceError):
            _launch([d], *bad)
    d.beta = 1.0
    with pytest.raises(L.GrassmannDeviceError):
        _launch([d], "f64", "f64", 64, 0, 0, symmetric=1)


def test_the_report_names_the_kernel():
    from grassmanntn_amd import _lib as L
    from grassmanntn_amd._device import DeviceArray
    from grassmanntn_amd.core import _gemm, _gemm_desc
    lib = L.lib()
    lib.gtn_autotune_set(1)
    x, y = DeviceArray.zeros((448, 448)), DeviceArray.zeros((448, 448))
    _gemm([_gemm_desc(x.data_ptr(), 448, 1, x.data_ptr(), 448, 1, y.data_ptr(), 448, 1, 448, 448, 448)], L.GTN_F64, "f64")
    n = lib.gtn_autotune_report(None, 0)
    arr = (L.TuneEntry * n)()
    lib.gtn_autotune_report(arr, n)
    mine = [e for e in arr if (e.M, e.N, e.K, e.batch) == (448, 448, 448, 1)]
    assert mine and all(e.kernel in (0, 1) for e in mine)
