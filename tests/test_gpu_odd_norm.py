"""gtn_odd_norm and the singular values' norms on the device, over shapes with and without the bit-mask parity."""
import numpy as np
import pytest

from oracle import gtn_oracle as O

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")


@pytest.mark.parametrize("stats,shape", [((1,), (1,)), ((1, -1), (2, 4)), ((0, 1, -1), (3, 4, 8)), ((1, 0, -1), (4, 3, 8)),
                                         ((1, -1, 0), (4, 4, 5)), ((1, 0, 0, -1), (8, 7, 9, 16)), ((0, 0), (3, 5)),
                                         ((1, 1, -1, -1), (32, 32, 32, 32))])
@pytest.mark.parametrize("pp", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128])
def test_odd_norm(stats, shape, pp, dtype):
    """Against the sum over the entries of odd parity; rounding of a sum of n squares in FP64."""
    from grassmanntn_amd import core
    rng = np.random.default_rng(sum(shape))
    X = rng.standard_normal(shape).astype(dtype)
    if dtype is np.complex128:
        X = X + 1j * rng.standard_normal(shape)
    T = gtn.dense(X, encoder="parity-preserving" if pp else "canonical", statistics=stats)
    par = np.zeros(shape, dtype=np.int64)
    for a, (d, s) in enumerate(zip(shape, stats)):
        if s:
            p = np.arange(d) & 1 if pp else O.parity_of_canonical(np.arange(d))
            par = par + p.reshape([-1 if b == a else 1 for b in range(len(shape))])
    ref = float(np.sum(np.abs(X.astype(np.complex128)) ** 2 * (par % 2)))
    assert abs(float(core._odd_norm_dev(T).item()) - ref) <= 1e-13 * max(ref, 1e-300)
