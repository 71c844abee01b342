"""GPU tests of gtn_svd_blocks at the sizes where its kernels' tiles and vector groups end: small
blocks (both sides at most 128: one-sided Jacobi on the block, 16 vectors per wavefront in groups of
eight, one or two components per lane), and the block width of the range finder (CholeskyQR in 16 x 16
tiles, Rayleigh-Ritz matrix) around multiples of 16.

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


@pytest.mark.parametrize("m,n", [(1, 1), (1, 5), (2, 2), (7, 5), (15, 16), (16, 16), (17, 15), (16, 33), (63, 64), (65, 64),
                                 (64, 128), (113, 112), (127, 128), (128, 127), (128, 128), (128, 129), (40, 300)])
def test_small_blocks(m, n):
    """Full decompositions of blocks with a side of at most 128, singular values over three decades."""
    rng = np.random.default_rng(1000 * m + n)
    M = rng.standard_normal((m, n)) * 10.0 ** (-1.5 * np.arange(m) / m)[:, None] * 10.0 ** (-1.5 * np.arange(n) / n)
    k = min(m, n)
    outs, counts = _run([(M, k)])
    _check(M, k, outs[0], counts[0])


@pytest.mark.parametrize("m,n,r", [(16, 16, 3), (32, 20, 20), (128, 128, 37), (100, 128, 16), (128, 128, 0)])
def test_small_blocks_of_low_rank(m, n, r):
    """Rank r (0: the zero block): the rank rule keeps r values, the rest is exactly zero."""
    rng = np.random.default_rng(m + n + r)
    M = rng.standard_normal((m, r)) @ rng.standard_normal((r, n)) / max(1, r)
    outs, counts = _run([(M, min(m, n))])
    _check(M, min(m, n), outs[0], counts[0], rank=r)
    assert np.all(outs[0][1].numpy()[r:] == 0.0)


@pytest.mark.parametrize("m,n", [(3, 128), (16, 100), (17, 128), (100, 17), (64, 65), (128, 128)])
def test_small_blocks_with_zero_repeated_and_graded_rows(m, n):
    """Shorter sides well below the longer one, rows graded over ten decades in no order, rows of zeros and
    rows that repeat: what the triangular factor of a small block is built from."""
    rng = np.random.default_rng(100 * m + n)
    M = rng.standard_normal((m, n)) * 10.0 ** rng.uniform(-10, 0, m)[:, None]
    M[m // 2] = 0.0
    M[m - 1] = M[0]
    r = m - 2 if m <= n else n
    outs, counts = _run([(M, min(m, n))])
    assert counts[0] == r
    u, s, v = (x.numpy() for x in outs[0][:3])
    ref = np.linalg.svd(M, compute_uv=False)
    np.testing.assert_allclose(s, ref, rtol=0, atol=1e-13 * ref[0])
    np.testing.assert_allclose((u * s) @ v, M, rtol=0, atol=1e-13 * ref[0])


@pytest.mark.parametrize("k", [1, 8, 9, 16, 24, 32, 33])
@pytest.mark.parametrize("spectrum", ["flat", "equal", "pairs", "edge", "cluster", "steep", "random"])
def test_few_values_of_small_blocks(k, spectrum):
    """Fewer values than half a block has, where the pairs behind them are left out towards the end: spectra
    without a gap behind the last value wanted, with equal values around it and with large ones hidden
    in vectors that all have smaller norms."""
    rng = np.random.default_rng(k)
    n = 128 if k > 16 else 96
    s = {"flat": 1.0 - 1e-3 * np.arange(n), "equal": np.ones(n), "pairs": 0.97 ** (np.arange(n) // 2 * 2.0),
         "edge": np.where(np.arange(n) < k, 1.0, 1.0 - 1e-9), "cluster": np.where(np.arange(n) < k // 2, 1.0, 0.5),
         "steep": 0.7 ** np.arange(n), "random": np.sort(rng.uniform(0, 1, n))[::-1]}[spectrum]
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    R, _ = np.linalg.qr(rng.standard_normal((n, n)))
    outs, counts = _run([((Q * s) @ R, k), (Q * s, k)])
    for M, o, c in zip(((Q * s) @ R, Q * s), outs, counts):
        _check(M, k, o, c)


def test_small_blocks_scaled_and_repeated():
    """Entries far from one in magnitude, and values that coincide (a scaled orthogonal block)."""
    rng = np.random.default_rng(5)
    Q, _ = np.linalg.qr(rng.standard_normal((48, 48)))
    for M in (1e-120 * rng.standard_normal((48, 48)), 1e120 * rng.standard_normal((30, 48)), 3.0 * Q):
        outs, counts = _run([(M, 20)])
        s = outs[0][1].numpy()
        ref = np.linalg.svd(M, compute_uv=False)
        if ref[0] < 1e-28:  # the rank rule, sigma / (sigma_0 + 1e-14) > 1e-14, keeps nothing
            assert counts[0] == 0 and np.all(s == 0.0)
            continue
        np.testing.assert_allclose(s[:20], ref[:20], rtol=0, atol=1e-13 * ref[0])
        u = outs[0][0].numpy()[:, :20]
        np.testing.assert_allclose(u.T @ u, np.eye(20), rtol=0, atol=1e-13)


def test_mixed_batch_of_small_and_large_blocks():
    """One call over blocks of several shapes: more runs than one launch of the Jacobi kernel takes,
    the small ones of them in groups of equal shape."""
    rng = np.random.default_rng(8)
    blocks = []
    for i, (m, n, k) in enumerate([(8, 8, 4), (8, 8, 4), (20, 12, 6), (33, 33, 9), (5, 40, 5), (128, 100, 30), (140, 150, 10),
                                   (64, 64, 64), (3, 2, 1), (17, 17, 17), (140, 150, 10), (31, 47, 11), (96, 96, 2)]):
        w = 10.0 ** (-2.0 * np.arange(n) / n)
        blocks.append((rng.standard_normal((m, n)) * w, k))
    outs, counts = _run(blocks)
    for (M, k), o, c in zip(blocks, outs, counts):
        _check(M, k, o, c, tol=2e-13)


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

def _decaying_blocks(rng, m, n, s, count):
    blocks = []
    for _ in range(count):
        U, _r = np.linalg.qr(rng.standard_normal((m, m)))
        V, _r = np.linalg.qr(rng.standard_normal((n, m)))
        blocks.append((U * s) @ V.T)
    return blocks


@pytest.mark.parametrize("iters", [1, 2, 3, 4, 7, 20, 45])
@pytest.mark.parametrize("rate", [0.9, 0.96, 0.985])
def test_filtered_range_finder_is_no_further_off_than_plain_products(iters, rate):
    """The Gram iteration's filter against the alternating products M^T Y, M Z of the same count: every
    value within the bound that as many plain products give, (sigma_{p+1} / sigma_j)^(4 iters + 2) of it
    (the error of a Ritz value is quadratic in the missing part of its vector; a Gaussian start of
    p = 128 of 260 directions misses at most ~1e2 of it), plus rounding."""
    rng = np.random.default_rng(iters)
    k, p, m = 32, 128, 260
    s = rate ** np.arange(m)
    from grassmanntn_amd.core import settings
    blocks = [(M, k) for M in _decaying_blocks(rng, m, 300, s, 2)]
    old = settings.svd_iters
    settings.svd_iters = iters
    try:
        with gtn.precision("f64", "f64_gram"):
            outs, counts = _run(blocks)
    finally:
        settings.svd_iters = old
    miss = 1e4 * (s[p] / s[:k]) ** (4 * iters + 2)
    for (M, _k), o, c in zip(blocks, outs, counts):
        ref = np.linalg.svd(M, compute_uv=False)[:k]
        got = o[1].numpy()[:k]
        assert c == k
        assert np.all(got <= ref * (1 + 1e-13))
        assert np.all(ref - got <= (miss + 1e-13) * ref[0]), (np.max((ref - got) / ref[0]), miss.max())


@pytest.mark.parametrize("case", ["wide", "dropped", "low rank", "flat", "mixed"])
def test_filtered_range_finder_special_spectra(case):
    """Spectra at the rules' edges, several in one call: kept values near CholeskyQR's floor, directions
    under it, rank below k, no gap at all, and blocks that stop at different products."""
    rng = np.random.default_rng(11)
    m, k = 260, 24
    i = np.arange(m)
    spectra = {"wide": 10.0 ** (-3.2 * np.minimum(i, 60) / 60.0) * np.where(i < 60, 1.0, 0.3),
               "dropped": np.where(i < 40, 10.0 ** (-6.0 * i / 40), 0.0),
               "low rank": np.where(i < 9, 0.7 ** i, 0.0),
               "flat": np.ones(m)}
    names = ["wide", "low rank", "dropped", "flat"] if case == "mixed" else [case, case]
    blocks = [(_decaying_blocks(rng, m, 300, spectra[n], 1)[0], k) for n in names]
    outs, counts = _run(blocks)
    for name, (M, _k), o, c in zip(names, blocks, outs, counts):
        ref = np.linalg.svd(M, compute_uv=False)
        s = o[1].numpy()[:k]
        u = o[0].numpy()[:, :c]
        if name == "low rank":
            assert c == 9
        elif name == "dropped":
            assert c >= np.count_nonzero(ref[:k] > 1e-3)
        else:
            assert c == k
        np.testing.assert_allclose(s[:c], ref[:c], rtol=0, atol=(1e-12 if name == "flat" else 1e-13) * ref[0])
        np.testing.assert_allclose(u.T @ u, np.eye(c), rtol=0, atol=1e-13)


@pytest.mark.parametrize("m,n", [(129, 129), (191, 200), (192, 1000), (193, 193), (256, 257), (257, 2100), (383, 384)])
def test_gram_matrix_tiles(m, n):
    """Gram matrices whose size is around multiples of the 64 and 128 tiles, with short and long
    reductions (split into chunks), through decompositions of a single block: the values to rounding."""
    rng = np.random.default_rng(m)
    s = np.maximum(0.6 ** np.arange(m), 1e-3 * 0.97 ** np.arange(m))
    M = _decaying_blocks(rng, m, n, s, 1)[0]
    outs, counts = _run([(M, 12)])
    _check(M, 12, outs[0], counts[0])
