"""Workloads that stand for the use of grassmanntn_amd: coarse-graining steps of single tensors, of
batches and of whole coupling sweeps, the standalone tensor operations they are made of, and the
surrogate's training pass.  `listed` names one case of each; `draw` gives others of the same ranges.

Inputs are Grassmann-even tensors whose legs carry bond weights: a leg of a coarse-grained tensor is
an SVD bond, its entries scale with the square root of the kept singular values, and the kept values
of a late step fall to about 0.0085 of the largest.
"""
import math

import numpy as np
import torch

import grassmanntn_amd as gtn
from grassmanntn_amd._device import DeviceArray
from grassmanntn_amd.batch import BatchedTRG
from grassmanntn_amd.surrogate import MLPEnsemble
from grassmanntn_amd.sweep import CouplingSweep

EDGE = 0.0085  # smallest kept singular value of a late step over the largest
CHIS = (16, 24, 32, 48, 64)
SITE = (1, 1, -1, -1)


def listed():
    return [
        # one step of a small tensor: the latency of a single coarse-graining call
        {"name": "trg_d16", "kind": "trg", "D": 16, "chi": 16},
        # one step at the working size of a single tensor
        {"name": "trg_d64", "kind": "trg", "D": 64, "chi": 64},
        # the anisotropic step: four decompositions that follow one another
        {"name": "atrg_d32", "kind": "atrg", "D": 32, "chi": 24},
        # eight points advanced together by recorded steps at the working size
        {"name": "batch_d64", "kind": "batch", "D": 64, "chi": 64, "points": 8, "steps": 2},
        # a whole coupling sweep over uneven bond dimensions
        {"name": "sweep", "kind": "sweep", "D": 32, "points": 30, "steps": 6},
        # a contraction so small that only its latency counts
        {"name": "einsum_d8", "kind": "einsum", "D": 8, "arith": "f64", "dtype": "f64", "boson": 0},
        # the standalone contraction of two 64^4 tensors
        {"name": "einsum_d64", "kind": "einsum", "D": 64, "arith": "f64", "dtype": "f64", "boson": 0},
        # the same in the arithmetic of the mixed-precision schedule's later steps
        {"name": "einsum_f32_d64", "kind": "einsum", "D": 64, "arith": "f32", "dtype": "f64", "boson": 0},
        # FP32 tensors with odd bosonic legs (flavours, a free and a contracted one)
        {"name": "einsum_ragged", "kind": "einsum", "D": 32, "arith": "f32", "dtype": "f32", "boson": 3},
        # leg permutation, encoder switch and leg fusion of a working-size tensor
        {"name": "relayout_d64", "kind": "relayout", "D": 64, "boson": 1},
        # truncated decomposition with bosonic legs (the split of a three-dimensional site tensor)
        {"name": "svd_ragged", "kind": "svd", "D": 16, "boson": 5, "chi": 50},
        # forward and backward pass of the surrogate's ensemble over one training set
        {"name": "mlp_pass", "kind": "mlp", "rows": 4096, "width": 256, "members": 5},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("trg", "trg", "atrg", "batch", "sweep", "einsum", "einsum", "einsum", "relayout", "svd", "mlp"))
    if kind == "trg":
        D = rng.choice((4, 8, 16, 32, 64))
        return {"kind": kind, "D": D, "chi": rng.randint(max(4, D // 2), D)}
    if kind == "atrg":
        D = rng.choice((8, 16, 32))
        return {"kind": kind, "D": D, "chi": rng.randint(D // 2, D)}
    if kind == "batch":
        D = rng.choice((16, 32, 32, 64))
        return {"kind": kind, "D": D, "chi": rng.randint(D // 2, D), "points": rng.randint(2, 8), "steps": rng.randint(1, 2)}
    if kind == "sweep":
        return {"kind": kind, "D": rng.choice((16, 32)), "points": rng.randint(5, 30), "steps": rng.randint(4, 6)}
    if kind == "einsum":
        D = rng.choice((4, 8, 16, 32, 64))
        dtype, arith = rng.choice((("f64", "f64"), ("f64", "f64"), ("f64", "f32"), ("f32", "f32")))
        return {"kind": kind, "D": D, "arith": arith, "dtype": dtype, "boson": rng.choice((0, 3, 5, 7)) if D <= 32 else 0}
    if kind == "relayout":
        D = rng.choice((8, 16, 32, 64))
        return {"kind": kind, "D": D, "boson": rng.randint(1, 9) if D <= 32 else 1}
    if kind == "svd":
        return {"kind": kind, "D": rng.choice((4, 8, 16)), "boson": rng.randint(1, 7), "chi": rng.randint(6, 60)}
    return {"kind": kind, "rows": log_int(100, 8192), "width": rng.choice((64, 128, 200, 256)), "members": rng.randint(2, 6)}


# ---- inputs -------------------------------------------------------------------------------------
def _weights(d, stat):
    """Bond weights of a leg of d entries, sqrt of singular values falling to EDGE; the two parities
    of a fermionic leg share them."""
    r = np.arange(d) // (2 if stat else 1)
    return np.exp(0.5 * math.log(EDGE) * r / max(1, r[-1])).astype(np.float32)


def _tensor(rng, shape, stats):
    """Even tensor in the parity-preserving encoder (the parity is the index's lowest bit)."""
    X = rng.standard_normal(shape, dtype=np.float32)
    for a, (d, s) in enumerate(zip(shape, stats)):
        X *= _weights(d, s).reshape([-1 if b == a else 1 for b in range(len(shape))])
    par = np.zeros((1,) * len(shape), dtype=np.int8)
    for a, (d, s) in enumerate(zip(shape, stats)):
        if s:
            par = par ^ (np.arange(d, dtype=np.int8) & 1).reshape([-1 if b == a else 1 for b in range(len(shape))])
    X *= par == 0
    return X.astype(np.float64) / float(np.abs(X).max())


def _dense(X, stats):
    return gtn.dense(X, encoder="parity-preserving", statistics=stats)


def _pattern(case):
    """(subscripts, statistics and shapes of both operands) of an einsum case."""
    D, n = case["D"], case["boson"]
    if not n:
        return "ijkl,klmn->ijmn", SITE, (D,) * 4, SITE, (D,) * 4
    # a free flavour on the first operand, a contracted one on both, as in "iIaj,jIbk->akbi"
    return "iIaj,jIbk->akbi", (1, 0, -1, 1), (D, n, D, D), (-1, 0, 1, 1), (D, n, D, D)


def _arrays(case, seed):
    rng = np.random.default_rng(seed)
    kind, D = case["kind"], case.get("D")
    if kind == "trg":
        return [(_tensor(rng, (D,) * 4, SITE), SITE)]
    if kind == "atrg":
        return [(_tensor(rng, (D,) * 4, SITE), SITE) for _ in range(2)]
    if kind == "einsum":
        _, sa, xa, sb, xb = _pattern(case)
        ops = [(_tensor(rng, xa, sa), sa), (_tensor(rng, xb, sb), sb)]
        return [(x.astype(np.float32), s) for x, s in ops] if case["dtype"] == "f32" else ops
    if kind == "relayout":
        n = case["boson"]
        st = SITE + ((0,) if n > 1 else ())
        return [(_tensor(rng, (D,) * 4 + ((n,) if n > 1 else ()), st), st)]
    if kind == "svd":
        n, st = case["boson"], (1, -1, 0, 0, 1, -1)
        return [(_tensor(rng, (D, D, n, n, D, D), st), st)]
    raise ValueError(kind)


class _Kept:
    """What a program keeps between calls; its recorded graphs and their memory go with it."""

    def __init__(self, owner, **kw):
        self.owner = owner
        self.__dict__.update(kw)

    def __del__(self):
        self.owner.close()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        rng = np.random.default_rng(seed)
        T0 = np.stack([_tensor(rng, (case["D"],) * 4, SITE) for _ in range(case["points"])])
        T0 = DeviceArray.from_numpy(T0.reshape(case["points"], -1))
        run_ = BatchedTRG(case["points"], case["D"], case["chi"], case["steps"])
        run_.prepare(T0)
        return case, _Kept(run_, T0=T0)
    if kind == "sweep":
        rng = np.random.default_rng(seed)
        n = case["points"]
        beta, m = rng.uniform(0.1, 2.0, n), rng.uniform(0.0, 1.0, n)
        chi = np.resize([c for c in CHIS if c <= 2 * case["D"]], n)
        sw = CouplingSweep(case["D"], case["steps"])
        sw.prepare(beta, m, chi)
        return case, _Kept(sw, points=(beta, m, chi))
    if kind == "mlp":
        ens = MLPEnsemble((2,) + (case["width"],) * 3 + (17,), case["members"], seed)
        return case, (ens,) + tuple(DeviceArray.from_numpy(x) for x in _training_set(case, seed))
    return case, [_dense(x, s) for x, s in _arrays(case, seed)]


def _training_set(case, seed):
    rng = np.random.default_rng(seed)
    X = rng.uniform(-1.7, 1.7, (case["rows"], 2)).astype(np.float32)
    Y = rng.standard_normal((case["rows"], 17)).astype(np.float32)
    w = np.ones(17, dtype=np.float32)
    w[0] = 8.0
    return X, Y, w / w.sum()


# ---- one pass -----------------------------------------------------------------------------------
class _Shared:
    """A device array of the library offered to torch without a copy."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = {"shape": a.shape, "typestr": a.dtype.str, "data": (a.data_ptr(), False),
                                         "strides": None, "version": 2}


def _view(a):
    return torch.as_tensor(_Shared(a), device="cuda")


def run(state):
    case, s = state
    kind = case["kind"]
    if kind == "trg":
        T, nrm = gtn.trg(s[0], case["chi"])
        return {"T": _view(T.data), "norm": nrm}
    if kind == "atrg":
        T, nrm = gtn.atrg2dy(s[0], s[1], case["chi"])
        return {"T": _view(T.data), "norm": nrm}
    if kind == "batch":
        lnz = s.owner.run(s.T0)
        return {"T": _view(s.owner.xs), "lnz": lnz, "log_norms": s.owner.log_norms}
    if kind == "sweep":
        return {"lnz": s.owner.run(*s.points)}
    if kind == "einsum":
        with gtn.precision(case["arith"]):
            return {"C": _view(gtn.einsum(_pattern(case)[0], s[0], s[1]).data)}
    if kind == "relayout":
        T, tail = s[0], "" if case["boson"] == 1 else "n"
        P = gtn.einsum("ijkl%s->jkli%s" % (tail, tail), T)
        J = T.join_legs("(ij)(kl)" + tail, "matrix", intermediate_stat=(-1, 1) + ((0,) if tail else ()))
        return {"permuted": _view(P.data), "canonical": _view(T.switch_encoder().data), "joined": _view(J.data)}
    if kind == "svd":
        U, S, V = s[0].svd("(i a m)(n j b)", case["chi"])
        return {"U": _view(U.data), "S": _view(S.data), "V": _view(V.data)}
    ens, X, Y, w = s
    out = ens.forward(X)
    ens.backward(X, ens.loss_grad(out, Y, w))
    return {"out": _view(out), "grads": _view(ens.grads), "loss": _view(ens.loss)}


# ---- bytes and operations that a pass cannot do without --------------------------------------------
def _bond(chi, most):
    k = min(most, chi // 2)
    return 2 << max(0, math.ceil(math.log2(max(1, k)))) if k > 1 else 2


def _trg_work(D, chi):
    d = _bond(chi, D * D // 2)
    # T' and the two three-leg contractions; the projections of the four parity blocks
    return 8.0 * (D ** 4 + d ** 4), d ** 4 * D ** 2 / 2 + d ** 2 * D ** 3 + 2.0 * D ** 4 * d


def work(case):
    kind, D = case["kind"], case.get("D")
    if kind == "trg":
        b, f = _trg_work(D, case["chi"])
    elif kind == "atrg":
        d = _bond(case["chi"], D * D // 2)
        b = 8.0 * (2 * D ** 4 + d ** 4)
        f = (2.0 * D ** 4 * d + d ** 2 * D ** 3 / 2 + (D * d) ** 2 * d + 1.0 * D ** 2 * d ** 3
             + D ** 4 * d ** 2 / 2 + D ** 4 * d + d ** 3 * D ** 2 / 2)
    elif kind == "batch":
        b1, f1 = _trg_work(D, case["chi"])
        d = _bond(case["chi"], D * D // 2)
        b2, f2 = _trg_work(d, case["chi"])
        n = case["points"]
        b, f = n * (b1 + (case["steps"] - 1) * b2), n * (f1 + (case["steps"] - 1) * f2)
    elif kind == "sweep":
        b = f = 0.0
        for c in np.resize([c for c in CHIS if c <= 2 * D], case["points"]):
            d = _bond(int(c), D * D // 2)
            b1, f1 = _trg_work(D, int(c))
            b2, f2 = _trg_work(d, int(c))
            b, f = b + b1 + (case["steps"] - 1) * b2, f + f1 + (case["steps"] - 1) * f2
    elif kind == "einsum":
        n, es = max(1, case["boson"]), 8.0 if case["dtype"] == "f64" else 4.0
        b = es * (2 * n * D ** 3 + D ** 4) if case["boson"] else es * 3 * D ** 4
        f = n * D ** 5 / 2.0 if case["boson"] else D ** 6 / 2.0
    elif kind == "relayout":
        b, f = 8.0 * 4 * D ** 4 * case["boson"], 0.0
    elif kind == "svd":
        m, n = D * D * case["boson"], D * D * case["boson"]
        d = _bond(case["chi"], m // 2)
        b, f = 8.0 * (m * n + (m + n) * d + d * d), 2.0 * (m / 2.0) * n * d
    else:
        h, e, r = case["width"], case["members"], case["rows"]
        params = 2 * h + 2 * h * h + 17 * h
        b, f = 4.0 * (e * params * 2 + r * 19 + e * r * 17), 6.0 * e * r * params
    return {"bytes": b, "flops": f}


# ---- the same in 64 bits -------------------------------------------------------------------------
def _popcount(x):
    return np.array([bin(int(v)).count("1") for v in x])


def _canonical(d):
    """Canonical index of each parity-preserving index: its lowest bit makes the popcount's parity
    that of the index."""
    i = np.arange(d)
    return i ^ (_popcount(i >> 1) & 1)


def _sigma(d):
    """(-1)^(p (p - 1) / 2) of each parity-preserving index, p its occupation."""
    return np.where(_popcount(_canonical(d)) % 4 >= 2, -1.0, 1.0)


def _inversions(a, b, odd):
    pos = {c: k for k, c in enumerate(b)}
    o = [pos[c] for c in a if odd[c]]
    return sum(o[x] > o[y] for x in range(len(o)) for y in range(x + 1, len(o))) & 1


def _grassmann(sub, *ops):
    """Grassmann einsum of (tensor, statistics) pairs in the parity-preserving encoder: one plain
    contraction for each pattern of the fermionic parities, with the sign of bringing every contracted
    pair together and of ordering the rest as in the output."""
    ins, out = sub.split("->")
    ins = ins.split(",")
    chars, stats = "".join(ins), [s for _, st in ops for s in st]
    dim = {c: d for s, (X, _) in zip(ins, ops) for c, d in zip(s, X.shape)}
    ferm = [c for c in dict.fromkeys(chars) if any(s for x, s in zip(chars, stats) if x == c)]
    pairs = [c for c in ferm if chars.count(c) > 1]
    seq = [c.upper() + "*" if (s < 0 and c in pairs) else c for c, s in zip(chars, stats) if s]
    kept = [c for c in seq if not c.endswith("*")]
    moved = [x for c in kept for x in ([c, c.upper() + "*"] if c in pairs else [c])]
    rest = [c for c in kept if c not in pairs]
    fout = [c for c in out if c in ferm]
    first = ops[0][0]
    res = torch.zeros([dim[c] for c in out], dtype=torch.float64, device=first.device)
    sig = {c: torch.as_tensor(_sigma(dim[c]), device=first.device) for c in pairs}
    for m in range(1 << len(ferm)):
        odd = {c: (m >> k) & 1 for k, c in enumerate(ferm)}
        if any(sum(odd[c] for c in s if c in odd) & 1 for s in ins):
            continue
        par = dict(odd, **{c.upper() + "*": odd[c] for c in pairs})
        sign = -1.0 if _inversions(seq, moved, par) ^ _inversions(rest, fout, par) else 1.0
        cut = lambda s, X: X[tuple(slice(odd[c], None, 2) if c in odd else slice(None) for c in s)]  # noqa: E731
        parts = [cut(s, X) for s, (X, _) in zip(ins, ops)]
        terms, names = list(parts), list(ins)
        if len(ops) > 1:
            for c in pairs:  # each contracted index once, on the first operand that has it
                s = names[0]
                terms[0] = terms[0] * sig[c][odd[c]::2].reshape([-1 if x == c else 1 for x in s])
        cut(out, res).add_(torch.einsum(",".join(names) + "->" + out, *[t.contiguous() for t in terms]), alpha=sign)
    return res


def _split(T, stats, chi):
    """(U, S, V) of the fused matrix of a four-leg tensor's first and last two legs, int(chi / 2)
    values in each parity block, every column of U with its largest entry positive."""
    a, b = T.shape[0], T.shape[1]
    can = (_canonical(a)[:, None] * b + _canonical(b)[None, :]).reshape(-1)
    pop = _popcount(can)
    row = np.where(pop % 4 >= 2, -1.0, 1.0).reshape(a, b)
    for ax, s in enumerate(stats[:2]):
        if s == 1:
            row = row * np.where(np.arange(T.shape[ax]) & 1, -1.0, 1.0).reshape([-1, 1] if ax == 0 else [1, -1])
    row = row.reshape(-1)
    colpar = (_popcount((_canonical(T.shape[2])[:, None] * T.shape[3] + _canonical(T.shape[3])[None, :]).reshape(-1)) & 1)
    M = T.reshape(a * b, -1) * row[:, None]
    keep = []
    for p in (0, 1):
        r, c = np.nonzero((pop & 1) == p)[0], np.nonzero(colpar == p)[0]
        U, s, V = np.linalg.svd(M[np.ix_(r, c)], full_matrices=False)
        k = min(int(np.sum(s / (s[0] + 1e-14) > 1e-14)), chi // 2)
        sg = np.sign(U[np.argmax(np.abs(U[:, :k]), axis=0), np.arange(k)])
        keep.append((r, c, U[:, :k] * sg, s[:k], V[:k] * sg[:, None]))
    d = max(len(x[3]) for x in keep)
    d = 2 ** math.ceil(math.log2(d)) if d > 1 else 1
    U, S, V = np.zeros((a * b, 2 * d)), np.zeros(2 * d), np.zeros((2 * d, M.shape[1]))
    for p, (r, c, u, s, v) in enumerate(keep):
        k = len(s)
        at = 2 * np.arange(k) + p
        U[np.ix_(r, at)], S[at], V[np.ix_(at, c)] = u, s, v
    sx = _sigma(2 * d)
    return (U * row[:, None]).reshape(a, b, 2 * d), np.diag(S * sx), np.diag(np.sqrt(np.where(S > 1e-10, S, 0.0)) * sx), \
        (V * sx[:, None]).reshape((2 * d,) + T.shape[2:])


def _exact_trg(T, chi):
    def e(sub, *ops):
        return _grassmann(sub, *[(torch.as_tensor(X), st) for X, st in ops]).numpy()

    T1, T2 = e("ijkl->jkli", (T, SITE)), e("ijkl->klij", (T, SITE))
    s1, s2 = (1, -1, -1, 1), (-1, -1, 1, 1)
    U1, _, r1, V1 = _split(T1, s1, chi)
    U2, _, r2, V2 = _split(T2, s2, chi)
    U1, V1 = e("abx,xc->abc", (U1, s1[:2] + (1,)), (r1, (-1, 1))), e("ax,xbc->abc", (r1, (-1, 1)), (V1, (-1,) + s1[2:]))
    U2, V2 = e("abx,xc->abc", (U2, s2[:2] + (1,)), (r2, (-1, 1))), e("ax,xbc->abc", (r2, (-1, 1)), (V2, (-1,) + s2[2:]))
    VV = e("kwz,lxw->lxzk", (V1, (-1, -1, 1)), (V2, (-1, 1, 1)))
    UU = e("yxi,zyj->jzxi", (U1, (1, -1, 1)), (U2, (-1, -1, 1)))
    R = e("lxzk,jzxi->ijkl", (VV, (-1, 1, 1, -1)), (UU, (1, -1, -1, 1)))
    n = float(np.linalg.norm(R))
    return {"T": R / n, "norm": n}


def _exact_mlp(case, seed):
    X, Y, w = (torch.as_tensor(x.astype(np.float64)) for x in _training_set(case, seed))
    dims, e = (2,) + (case["width"],) * 3 + (17,), case["members"]
    Ws = [[] for _ in range(4)]
    for k in range(e):
        rng = np.random.default_rng(seed * 1000003 + k)
        for l in range(4):
            Ws[l].append((rng.standard_normal((dims[l], dims[l + 1])) * np.sqrt(1.0 / dims[l])).astype(np.float32))
    Ws = [torch.as_tensor(np.stack(x).astype(np.float64)).requires_grad_() for x in Ws]
    bs = [torch.zeros((e, dims[l + 1]), dtype=torch.float64, requires_grad=True) for l in range(4)]
    H = X[None].expand(e, -1, -1)
    for l in range(4):
        H = torch.matmul(H, Ws[l]) + bs[l][:, None, :]
        H = torch.nn.functional.gelu(H) if l < 3 else H
    loss = (w * (H - Y) ** 2).sum(dim=(1, 2)) / case["rows"]
    loss.sum().backward()
    grads = torch.cat([t.grad.reshape(-1) for l in range(4) for t in (Ws[l], bs[l])])
    return {"out": H.detach(), "grads": grads, "loss": loss.detach()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "trg":
        return _exact_trg(_arrays(case, seed)[0][0], case["chi"]) if case["D"] <= 32 else None
    if kind == "einsum":
        dev = "cuda" if torch.cuda.is_available() and case["D"] > 16 else "cpu"
        ops = [(torch.as_tensor(x.astype(np.float64), device=dev), s) for x, s in _arrays(case, seed)]
        return {"C": _grassmann(_pattern(case)[0], *ops)}
    if kind == "relayout":
        X, st = _arrays(case, seed)[0]
        tail = "n" if len(st) == 5 else ""
        P = _grassmann("ijkl%s->jkli%s" % (tail, tail), (torch.as_tensor(X), st)).numpy()
        can = [_canonical(d) for d in X.shape[:4]]
        C = np.empty_like(X)
        C[np.ix_(*can)] = X
        D = X.shape[0]
        # fused first pair: (-1)^p of both +1 legs and the matrix format's sigma
        pair = (can[0][:, None] * D + can[1][None, :]).reshape(-1)
        pop = _popcount(pair)
        sign = np.where(pop % 4 >= 2, -1.0, 1.0) * np.where(pop & 1, -1.0, 1.0)
        where = pair ^ (_popcount(pair >> 1) & 1)
        J = np.empty((D * D, D * D) + X.shape[4:])
        J[np.ix_(where, where)] = (X.reshape((D * D, D * D) + X.shape[4:]).T * sign).T
        return {"permuted": P, "canonical": C, "joined": J}
    if kind == "mlp":
        return _exact_mlp(case, seed)
    return None
