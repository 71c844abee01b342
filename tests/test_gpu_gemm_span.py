"""Products of operands whose slab ends on the last bytes of the 2 GiB that a buffer resource spans: 64 rows
whose last element begins one element below 2^31 bytes from the first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")


@pytest.mark.parametrize("dtype,k", [("f64", 16), ("f32", 32)])
@pytest.mark.parametrize("side", ["a", "b"])
def test_slab_of_two_gibibytes(dtype, k, side):
    """Small integers: the products are exact."""
    from grassmanntn_amd import _lib as L
    from grassmanntn_amd._device import DeviceArray
    from grassmanntn_amd.core import _gemm, _gemm_desc
    npd = np.float64 if dtype == "f64" else np.float32
    es = npd().itemsize
    elems = (1 << 31) // es
    ld = (elems - k) // 63
    assert 63 * ld + k == elems and ld * es % 16 == 0
    rng = np.random.default_rng(k)
    X, Y = rng.integers(1, 9, (64, k)), rng.integers(1, 9, (k, 64))
    wide = np.zeros(elems, dtype=npd)
    for r in range(64):
        wide[r * ld:r * ld + k] = X[r]
    dX, dY = DeviceArray.from_numpy(wide), DeviceArray.from_numpy(np.ascontiguousarray(Y.astype(npd)))
    dC = DeviceArray.zeros((64, 64), npd)
    if side == "a":
        d = _gemm_desc(dX.data_ptr(), ld, 1, dY.data_ptr(), 64, 1, dC.data_ptr(), 64, 1, 64, 64, k)
    else:  # the transposed product: the wide operand is B, contiguous along the reduction
        d = _gemm_desc(dY.data_ptr(), 1, 64, dX.data_ptr(), 1, ld, dC.data_ptr(), 64, 1, 64, 64, k)
    for _ in range(2):  # the autotuner's trials, then its choice
        _gemm([d], L.GTN_F64 if dtype == "f64" else L.GTN_F32, dtype)
        want = X @ Y
        assert np.array_equal(dC.numpy(), want if side == "a" else want.T)
