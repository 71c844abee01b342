"""GPU tests of gtn_svd_blocks at the sizes where its kernels' tiles end: the block width of the range
finder (CholeskyQR in 16 x 16 tiles) around multiples of 16.

Tolerances: a backward stable FP64 SVD moves a singular value by at most c eps sigma_0, c of the order
of the size: 1e-13 sigma_0 for 128, and the vectors' orthogonality and the reconstruction likewise.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")


def _run(blocks):
    from grassmanntn_amd import core
    from grassmanntn_amd._device import DeviceArray
    return core._svd_blocks_raw([(DeviceArray.from_numpy(M), k) for M, k in blocks], 0)


def _check(M, k, out, count, rank=None, tol=1e-13):
    u, s, v = (x.numpy() for x in out[:3])
    ref = np.linalg.svd(M, compute_uv=False)
    s0 = ref[0] if ref[0] > 0 else 1.0
    np.testing.assert_allclose(s[:k], ref[:k], rtol=0, atol=tol * s0)
    c = min(k, rank if rank is not None else k)
    assert count == c, (M.shape, count, c)
    u, s, v = u[:, :c], s[:c], v[:c]
    # the side the eigenvectors come from (small blocks: the shorter one; large ones: U), and the
    # other, M^T u / sigma or M v / sigma, whose angles see sigma_0 / sigma
    right = M.shape[0] > M.shape[1] and M.shape[1] <= 128
    e, x = (v @ v.T, u.T @ u) if right else (u.T @ u, v @ v.T)
    np.testing.assert_allclose(e, np.eye(c), rtol=0, atol=tol)
    np.testing.assert_allclose(x * s[:, None] * s[None, :], np.diag(s * s), rtol=0, atol=tol * s0 * s0)
    np.testing.assert_allclose(M @ v.T if right else (u.T @ M).T, (u * s) if right else (s[:, None] * v).T, rtol=0,
                               atol=tol * s0)
    assert np.all(np.diff(s) <= tol * s0)


@pytest.mark.parametrize("oversample", [3, 8, 9, 24, 25, 57, 89, 96])
def test_range_finder_widths(oversample):
    """Block widths p = k + oversample around multiples of 16 (odd ones are padded), 260 x 300 blocks
    whose values fall fast enough that twenty iterations converge at every width."""
    from grassmanntn_amd.core import settings
    rng = np.random.default_rng(oversample)
    k = 7
    blocks = []
    for _ in range(2):
        U, _r = np.linalg.qr(rng.standard_normal((260, 260)))
        V, _r = np.linalg.qr(rng.standard_normal((300, 260)))
        blocks.append(((U * np.maximum(0.55 ** np.arange(260), 1e-3 * 0.99 ** np.arange(260))) @ V.T, k))
    old = settings.svd_oversample
    settings.svd_oversample = oversample
    try:
        outs, counts = _run(blocks)
    finally:
        settings.svd_oversample = old
    for (M, kk), o, c in zip(blocks, outs, counts):
        _check(M, kk, o, c)


def test_non_finite_blocks_raise():
    from grassmanntn_amd import _lib as L
    rng = np.random.default_rng(3)
    for bad in (np.nan, np.inf):
        for m, n in ((20, 20), (128, 128), (150, 150)):
            M = rng.standard_normal((m, n))
            M[m // 2, n // 3] = bad
            with pytest.raises(L.GrassmannDeviceError):
                _run([(M, 5)])
