"""The signed gather as include/gtn_hip.h defines it, element by element in numpy, over the builder of
grassmanntn_amd._perm; and random gathers over every form the builder has: fused and plain virtual axes
in either encoder, fused, split and plain source axes, sigmas, traced legs, bosonic (odd) extents."""
import numpy as np

from grassmanntn_amd._perm import Perm


def popcount(x):
    x = np.asarray(x, dtype=np.int64)
    c = np.zeros_like(x)
    while np.any(x):
        c += x & 1
        x = x >> 1
    return c


def enc(x):
    return x ^ (popcount(x >> 1) & 1)


def offsets(P):
    """(source offset, code) of every output element, C order; code 0: +1, 1: -1, 2: zero."""
    shape = P.out_shape()
    idx = np.indices(shape).reshape(len(shape), -1) if shape else np.zeros((0, 1), dtype=np.int64)
    n = idx.shape[1]
    V = [np.zeros(n, dtype=np.int64) for _ in P.virts]
    for a, (_dim, feeds) in enumerate(P.outs):
        for v, mul in feeds:
            V[v] += idx[a] * mul
    F = [np.zeros(n, dtype=np.int64) for _ in P.ins]
    neg = np.zeros(n, dtype=np.int64)
    bits = np.zeros(n, dtype=np.int64)
    for v, (_dim, e, sig, comps) in enumerate(P.virts):
        c = enc(V[v]) if e else V[v]
        if sig:
            neg ^= (popcount(c) >> 1) & 1
        for cid in reversed(comps):
            dim, bit, csig, tg = P.comps[cid]
            k = c % dim
            c = c // dim
            pc = popcount(k)
            if bit >= 0:
                bits ^= (pc & 1) << bit
            if csig:
                neg ^= (pc >> 1) & 1
            for i, m in tg:
                F[i] += k * m
    off = np.zeros(n, dtype=np.int64)
    for b, (_dim, e, sig, split, st, lo) in enumerate(P.ins):
        if sig:
            neg ^= (popcount(F[b]) >> 1) & 1
        x = enc(F[b]) if e else F[b]
        off += (x & 1) * lo + (x >> 1) * st if split else x * st
    code = np.asarray(P.codes)[bits]
    return off, np.where(code == 2, 2, code ^ neg)


def gather(P, src, alpha=1.0):
    off, code = offsets(P)
    v = src.reshape(-1)[off].astype(np.float64) * np.where(code == 1, -alpha, alpha)
    return np.where(code == 2, 0.0, v).astype(src.dtype).reshape(P.out_shape())


def random_gather(rng, dims, odd=False, trace=False):
    """A random gather over legs of the given dimensions (powers of two; with odd=True some become
    bosonic extents of 3, 5 or 6 and are neither encoded nor fused with others), and its source size."""
    legs = []
    for d in dims:
        boson = odd and rng.random() < 0.4
        legs.append([int(rng.choice([3, 5, 6])) if boson else int(d), not boson])
    order = [int(x) for x in rng.permutation(len(legs))]

    def groups(seq):
        out, i = [], 0
        while i < len(seq):
            n = int(rng.integers(1, 3))
            g = seq[i:i + n]
            if not all(legs[x][1] for x in g):
                g = g[:1]
            out.append(g)
            i += len(g)
        return out

    P = Perm()
    # source: groups of legs fused into one axis each, in a random storage order
    src_groups = groups([int(x) for x in rng.permutation(len(legs))])
    axes, total = [], 1
    for g in reversed([src_groups[int(x)] for x in rng.permutation(len(src_groups))]):
        full = int(np.prod([legs[x][0] for x in g]))
        axes.append((g, full, total))
        total *= full
    feed = {}
    for g, full, stride in axes:
        fermi = all(legs[x][1] for x in g)
        split = fermi and full >= 4 and rng.random() < 0.3
        if split:  # even entries first, then the odd ones: half index at `stride`, parity half the axis on
            i = P.add_in(full, stride, enc=True, split=True, stride_lo=stride * (full // 2))
        else:
            i = P.add_in(full, stride, enc=fermi and rng.random() < 0.6, sigma=fermi and rng.random() < 0.2)
        m = full
        for x in g:
            m //= legs[x][0]
            feed[x] = [(i, m)]
    traced = -1
    if trace:
        cand = [x for x in range(len(legs)) if legs[x][1]]
        if cand:
            traced = cand[0]
            i = P.add_in(legs[traced][0], total, enc=bool(rng.random() < 0.5))
            total *= legs[traced][0]
            feed[traced].append((i, 1))
    nbit = 0
    for g in groups(order):
        fermi = all(legs[x][1] for x in g)
        full = int(np.prod([legs[x][0] for x in g]))
        v = P.add_virt(full, enc=fermi and rng.random() < 0.6, sigma=fermi and rng.random() < 0.2)
        for x in g:
            bit = -1
            if legs[x][1] and nbit < 7 and rng.random() < 0.8:
                bit = nbit
                nbit += 1
            P.add_comp(v, legs[x][0], feed[x], bit=bit, sigma=legs[x][1] and rng.random() < 0.2)
        if fermi and full >= 4 and rng.random() < 0.4:  # parity and half index as two output axes
            P.add_out(2, [(v, 1)])
            P.add_out(full // 2, [(v, 2)])
        else:
            P.add_out(full, [(v, 1)])
    codes = [int(x) for x in rng.choice([0, 1, 2], size=1 << nbit, p=[0.45, 0.45, 0.1])]
    P.set_table(codes)
    return P, total
