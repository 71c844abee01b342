"""Composed gathers (grassmanntn_amd._perm.compose) against their two steps, in numpy."""
import numpy as np
import pytest

from gather_reference import gather, random_gather
from grassmanntn_amd._perm import Perm, compose, strides


def _read_back(rng, inner, plain=True):
    """A gather over the tensor `inner` writes, its legs one source axis each: the operand gather of a
    contraction, two fused groups of legs in random order."""
    shape = inner.out_shape()
    P = Perm()
    st = strides(shape)
    ins = []
    for b, (n, s) in enumerate(zip(shape, st)):
        v = inner.outs[b][1][0][0]
        ins.append(P.add_in(n, s, enc=inner.virts[v][1] if plain else not inner.virts[v][1],
                            sigma=bool(rng.random() < 0.3) and n & (n - 1) == 0))
    order = [int(x) for x in rng.permutation(len(shape))]
    at, nbit = 0, 0
    while at < len(order):
        g = order[at:at + int(rng.integers(1, 3))]
        if any(shape[x] & (shape[x] - 1) for x in g):
            g = g[:1]
        at += len(g)
        full = int(np.prod([shape[x] for x in g]))
        fermi = full & (full - 1) == 0
        v = P.add_virt(full, enc=fermi and bool(rng.random() < 0.7))
        for x in g:
            P.add_comp(v, shape[x], [(ins[x], 1)], bit=nbit, sigma=fermi and bool(rng.random() < 0.3))
            nbit += 1
        P.add_out(full, [(v, 1)])
    P.set_table([int(x) for x in rng.choice([0, 1, 2], size=1 << nbit, p=[0.45, 0.45, 0.1])])
    return P


@pytest.mark.parametrize("seed", range(40))
def test_composed_gather_equals_its_two_steps(seed):
    rng = np.random.default_rng(seed)
    inner, n = random_gather(rng, rng.choice([2, 4, 8], size=4), odd=seed % 3 == 0)
    plain = all(len(f) == 1 and f[0][1] == 1 for _d, f in inner.outs) and all(len(v[3]) == 1 for v in inner.virts)
    outer = _read_back(rng, inner)
    src = rng.standard_normal(n)
    G = compose(outer, inner)
    assert (G is not None) == plain  # fused or halved axes in between do not compose
    if G is not None:
        assert np.array_equal(gather(G, src, 0.5), gather(outer, gather(inner, src), 0.5))


def test_composed_gather_refuses_other_encoders_and_traces():
    rng = np.random.default_rng(2)
    inner = Perm()
    i = inner.add_in(8, 1, enc=True)
    v = inner.add_virt(8, enc=True)
    inner.add_comp(v, 8, [(i, 1)], bit=0)
    inner.add_out(8, [(v, 1)])
    inner.set_table([0, 1])
    assert compose(_read_back(rng, inner), inner) is not None
    assert compose(_read_back(rng, inner, plain=False), inner) is None
    outer = Perm()
    a, b = outer.add_in(8, 1, enc=True), outer.add_in(8, 8, enc=True)
    v = outer.add_virt(8)
    outer.add_comp(v, 8, [(a, 1), (b, 1)])
    outer.add_out(8, [(v, 1)])
    assert compose(outer, inner) is None
