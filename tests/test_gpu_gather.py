"""gtn_permute bit for bit against its definition over random gathers: every table-driven path (row walk
in 256- and 1024-column chunks, LDS tiles, element walk; groups joined by addition or exclusive or) and
the descriptor walk, sizes from one element to beyond the largest chunk, F64 and F32."""
import numpy as np
import pytest

from gather_reference import gather, offsets, random_gather

pytestmark = pytest.mark.gpu

gtn = pytest.importorskip("grassmanntn_amd")


def _run(P, src, alpha):
    from grassmanntn_amd._device import DeviceArray
    return P.run(DeviceArray.from_numpy(src), alpha=alpha).numpy()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("sizes", [(1,), (2, 4), (4, 4, 4), (8, 8, 16), (16, 32, 16), (8, 8, 8, 8), (16, 16, 32, 16), (2, 64, 2, 128),
                                   (32, 16, 64, 64), (256, 8, 1024)])
def test_random_gathers(sizes, odd, dtype):
    for seed in range(6):
        rng = np.random.default_rng([seed, len(sizes), sizes[0], odd])
        P, n = random_gather(rng, sizes, odd=odd, trace=seed == 5 and np.prod(sizes) <= 1 << 16)
        src = rng.standard_normal(n).astype(dtype)
        assert offsets(P)[0].max() < n
        assert np.array_equal(_run(P, src, 1.0), gather(P, src, 1.0)), (sizes, seed)
        assert np.array_equal(_run(P, src, -0.5), gather(P, src, -0.5)), (sizes, seed)


def test_random_gathers_without_tables(monkeypatch):
    monkeypatch.setenv("GTN_PERM_NO_TABLES", "1")
    for seed in range(6):
        rng = np.random.default_rng(seed)
        P, n = random_gather(rng, (16, 32, 16), odd=seed % 2 == 1)
        src = rng.standard_normal(n)
        assert np.array_equal(_run(P, src, 1.0), gather(P, src, 1.0)), seed


@pytest.mark.parametrize("shape", [(32, 32, 16, 9), (64, 16, 5), (8, 1024, 3), (64, 7, 3, 5, 64), (16, 16, 3, 16, 3), (4, 2, 128, 15)])
@pytest.mark.parametrize("order", ["kept", "front", "reversed"])
def test_rows_of_odd_trailing_extents(shape, order):
    """Rows whose last axes are no powers of two (bosonic tails), in place and moved."""
    from grassmanntn_amd._perm import Perm, strides
    n = len(shape)
    perm = {"kept": list(range(n)), "front": [*range(1, n - 1), 0, n - 1], "reversed": list(range(n))[::-1]}[order]
    P = Perm()
    st = strides(shape)
    pow2 = [d & (d - 1) == 0 for d in shape]
    ins = [P.add_in(d, st[a], enc=pow2[a]) for a, d in enumerate(shape)]
    ferm = [a for a in perm if pow2[a]]
    for a in perm:
        v = P.add_virt(shape[a])
        P.add_comp(v, shape[a], [(ins[a], 1)], bit=ferm.index(a) if pow2[a] else -1, sigma=pow2[a])
        P.add_out(shape[a], [(v, 1)])
    P.set_table([(m * 7 >> 2) & 1 for m in range(1 << len(ferm))])
    src = np.random.default_rng(n).standard_normal(int(np.prod(shape)))
    assert np.array_equal(_run(P, src, -0.5), gather(P, src, -0.5))
