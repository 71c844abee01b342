"""The Gram iteration's filter (gtn_svd_blocks) against as many plain products of the same start: spectra
whose edge the first products estimate wrongly, where a count fixed by that estimate stops too early.

Tolerances: the filter's rules credit plain products with 1.2 times the ratio that they see, so what is left
in the kept space may not be further off than what plain products leave; a factor of four covers what
rounding makes of equal counts, and the floor is the rounding of m-term sums, 5e-13 at m of about 1000.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")

_Q = {}


def _block(s):
    """A len(s) x (len(s) + 36) block with singular values s (decreasing) in random bases."""
    m = len(s)
    if m not in _Q:
        rng = np.random.default_rng(m)
        _Q[m] = [np.linalg.qr(rng.standard_normal((m, m)))[0], np.linalg.qr(rng.standard_normal((m + 36, m)))[0]]
    U, V = _Q[m]
    return (U * s) @ V.T


def _errors(blocks, spectra, k, arithmetic):
    """Per block of one call: (error of the values, largest residual of M M^T u = sigma^2 u) over sigma_0 and its
    square."""
    from grassmanntn_amd import core
    from grassmanntn_amd._device import DeviceArray
    with gtn.precision("f64", arithmetic):
        outs, counts = core._svd_blocks_raw([(DeviceArray.from_numpy(M), k) for M in blocks], 0)
    res = []
    for M, s, o, c in zip(blocks, spectra, outs, counts):
        u, v = o[0].numpy()[:, :c], o[1].numpy()[:k]
        assert np.max(np.abs(u.T @ u - np.eye(c))) <= 1e-13
        r = M @ (M.T @ u) - u * v[:c] ** 2
        res.append((np.max(np.abs(v - s[:k])) / s[0], np.max(np.linalg.norm(r, axis=0)) / s[0] ** 2))
    return res


def _compare(spectra, k):
    blocks = [_block(s) for s in spectra]
    for plain, got in zip(_errors(blocks, spectra, k, "f64"), _errors(blocks, spectra, k, "f64_gram")):
        assert got[0] <= 4 * plain[0] + 5e-13 and got[1] <= 4 * plain[1] + 5e-13, (k, plain, got)


@pytest.mark.parametrize("k", [8, 32, 48, 64, 96, 112])
@pytest.mark.parametrize("rate", [0.9, 0.96, 0.98, 0.99, 0.995, 0.998, 0.999, 0.9995])
def test_geometric_spectra(k, rate):
    _compare([rate ** np.arange(1024)], k)


@pytest.mark.parametrize("k,top,step,n,tail", [
    # a plateau a little wider or narrower than the basis (p = 104, 112, 128) over a tail ...
    (16, 0, 1.0, 126, 0.44), (8, 0, 1.0, 114, 0.22), (8, 0, 1.0, 96, 0.45), (32, 0, 1.0, 138, 0.22), (32, 0, 1.0, 120, 0.1),
    (8, 0, 1.0, 140, 0.7), (64, 0, 1.0, 138, 0.45),
    # ... and the same under the values kept
    (8, 8, 0.55, 105, 0.45), (32, 32, 0.55, 129, 0.45), (32, 32, 0.77, 138, 0.45), (8, 8, 0.77, 96, 0.45), (32, 32, 0.3, 256, 0.2),
    (64, 64, 0.77, 138, 0.45)])
def test_plateaus(k, top, step, n, tail):
    """top values of 1, the rest of the first n at `step`, the others `tail` times that."""
    m = 700
    _compare([np.where(np.arange(m) < top, 1.0, np.where(np.arange(m) < n, step, step * tail))], k)


def test_blocks_that_start_and_stop_apart():
    """Several spectra of one shape in one call: the blocks filter from different products on."""
    i = np.arange(700)
    _compare([0.97 ** i, 0.999 ** i, np.where(i < 126, 1.0, 0.44), np.where(i < 9, 0.7 ** i, 0.0), np.maximum(0.8 ** i, 1e-7),
              np.where(i < 16, 1.0, np.where(i < 113, 0.5, 0.2))], 16)


@pytest.mark.parametrize("edges,levels", [((100, 131, 246, 294, 295), (1.0, 0.32, 0.17, 0.067, 0.026, 0.013)),
                                          ((100, 130, 222), (1.0, 0.393, 0.225, 0.177))])
def test_small_gaps_over_a_deep_tail(edges, levels):
    """A slow fall across the basis' width and steps behind it: the gap is small and the rest lies far below,
    so plain products bring it to rounding in a count that the filter's growth does not suffice in."""
    i = np.arange(700)
    _compare([np.asarray(levels)[np.searchsorted(edges, i, side="right")] * np.exp(-0.002 * i)], 8)
