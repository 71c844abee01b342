"""Builder for gtn_permute descriptors (the signed-gather kernel of include/gtn_hip.h).

A gather is described in terms of *components*: canonical indices of single legs.  Output raw
axes feed virtual axes (fused canonical or parity-preserving indices, possibly assembled from
several raw axes such as (parity, half-index)); virtual axes split into components; components
add into the fused indices of the source's axes.
"""
import ctypes as C
import functools

from . import _lib as L
from ._device import DeviceArray


class Perm:
    def __init__(self):
        self.outs = []    # (dim, [(virt, mul)])
        self.virts = []   # [dim, enc, sigma, [comp ids]]
        self.comps = []   # [dim, bit, sigma, [(in, mult)]]
        self.ins = []     # [dim, enc, sigma, split, stride, stride_lo]
        self.codes = [0]
        self.n_bits = 0
        self._descs = {}  # descriptors of the finished gather, by (dtype, source size, factor)

    def add_in(self, dim, stride, enc=False, sigma=False, split=False, stride_lo=0):
        self.ins.append([int(dim), bool(enc), bool(sigma), bool(split), int(stride), int(stride_lo)])
        return len(self.ins) - 1

    def add_virt(self, dim, enc=False, sigma=False):
        self.virts.append([int(dim), bool(enc), bool(sigma), []])
        return len(self.virts) - 1

    def add_comp(self, virt, dim, targets, bit=-1, sigma=False):
        """Append a component to `virt` (call in C order: most significant first)."""
        self.comps.append([int(dim), int(bit), bool(sigma), [(int(i), int(m)) for i, m in targets]])
        cid = len(self.comps) - 1
        self.virts[virt][3].append(cid)
        return cid

    def add_out(self, dim, feeds):
        self.outs.append((int(dim), [(int(v), int(m)) for v, m in feeds]))
        return len(self.outs) - 1

    def set_table(self, codes):
        n = max(0, (len(codes) - 1).bit_length())
        if len(codes) != (1 << n):
            raise ValueError("table length must be a power of two")
        self.codes = list(codes)
        self.n_bits = n

    def desc(self, dtype, src_elems, alpha=1.0):
        """The descriptor for one source; a gather that has been run is not built any further."""
        key = (dtype, src_elems, alpha)
        d = self._descs.get(key)
        if d is None:
            d = self._desc(dtype, src_elems, alpha)
            if len(self._descs) >= 8:
                self._descs = {}
            self._descs[key] = d
        return d

    def _desc(self, dtype, src_elems, alpha):
        d = L.PermDesc()
        if len(self.outs) > L.MAX_AX or len(self.virts) > L.MAX_AX or len(self.ins) > L.MAX_AX:
            raise NotImplementedError("gather with more than %d axes" % L.MAX_AX)
        if len(self.comps) > L.MAX_COMP:
            raise NotImplementedError("gather with more than %d legs" % L.MAX_COMP)
        d.dtype = dtype
        d.n_out, d.n_virt, d.n_in, d.n_bits = len(self.outs), len(self.virts), len(self.ins), self.n_bits
        for a, (dim, feeds) in enumerate(self.outs):
            d.out_dim[a] = dim
            d.out_virt[a][0] = d.out_virt[a][1] = -1
            for t, (v, m) in enumerate(feeds):
                d.out_virt[a][t] = v
                d.out_vmul[a][t] = m
        order = []
        for v, (dim, enc, sig, comps) in enumerate(self.virts):
            d.virt_dim[v] = dim
            d.virt_enc[v] = enc
            d.virt_sigma[v] = sig
            d.virt_ncomp[v] = len(comps)
            order += comps
        d.n_comp = len(order)
        for j, cid in enumerate(order):
            dim, bit, sig, tg = self.comps[cid]
            d.comp_dim[j] = dim
            d.comp_bit[j] = bit
            d.comp_sigma[j] = sig
            d.comp_in[j][0] = d.comp_in[j][1] = -1
            for t, (i, m) in enumerate(tg):
                d.comp_in[j][t] = i
                d.comp_mult[j][t] = m
        for b, (dim, enc, sig, split, st, stlo) in enumerate(self.ins):
            d.in_dim[b] = dim
            d.in_enc[b] = enc
            d.in_sigma[b] = sig
            d.in_split[b] = split
            d.in_stride[b] = st
            d.in_stride_lo[b] = stlo
        words = [0] * len(d.table)
        for m, code in enumerate(self.codes):
            words[m >> 4] |= (code & 3) << ((m & 15) * 2)
        for i, w in enumerate(words):
            d.table[i] = w
        if isinstance(alpha, complex):
            d.alpha_re, d.alpha_im = alpha.real, alpha.imag
        else:
            d.alpha_re, d.alpha_im = float(alpha), 0.0
        d.src_elems = int(src_elems)
        return d

    def out_shape(self):
        return tuple(dim for dim, _ in self.outs)

    def run(self, src, dst=None, alpha=1.0):
        """Launch on the current stream; returns dst (allocated when None)."""
        lib = L.lib()
        shape = self.out_shape()
        if dst is None:
            dst = DeviceArray.empty(shape, src.dtype)
        if dst.numel() == 0:
            return dst
        if not (src.is_contiguous() and dst.is_contiguous()):
            raise ValueError("gather operands must be contiguous")
        d = self.desc(L.dtype_code(src), src.numel(), alpha)
        L.check(lib.gtn_permute(C.byref(d), L.ptr(src), L.ptr(dst), L.stream_ptr()), "gtn_permute")
        return dst


@functools.lru_cache(maxsize=256)
def compose(outer, inner):
    """outer(inner(.)) as one gather, or None.  It is one when every axis between them carries a single
    leg: each source axis of `outer` is one component, unsplit, laid out as `inner` writes it, and each
    output axis of `inner` one component, read in the same encoder.  The legs of `outer` then feed what
    those of `inner` fed, and both sign tables join into one over their legs' parities."""
    shape = inner.out_shape()
    if len(outer.ins) != len(shape):
        return None
    feed = {}
    for cid, (dim, bit, sig, tg) in enumerate(outer.comps):
        if len(tg) != 1 or tg[0][1] != 1 or tg[0][0] in feed:
            return None
        feed[tg[0][0]] = cid
    through = {}
    for b, ((dim, enc, sig, split, st, _lo), n, want) in enumerate(zip(outer.ins, shape, strides(shape))):
        feeds = inner.outs[b][1]
        if b not in feed or split or dim != n or (st != want and n > 1) or len(feeds) != 1 or feeds[0][1] != 1:
            return None
        v = feeds[0][0]
        vdim, venc, vsig, vcomps = inner.virts[v]
        if vdim != n or venc != enc or len(vcomps) != 1 or v in through:
            return None
        through[v] = b
        cid = feed[b]
        if outer.comps[cid][0] != n:
            return None
    if len(through) != len(inner.virts):
        return None
    G = Perm()
    G.ins = [list(x) for x in inner.ins]
    G.outs = list(outer.outs)
    G.virts = [[d, e, sg, list(c)] for d, e, sg, c in outer.virts]
    of_outer, of_inner, comps = [], [], []
    for cid, (dim, bit, sig, tg) in enumerate(outer.comps):
        b = tg[0][0]
        icid = inner.virts[inner.outs[b][1][0][0]][3][0]
        _d, ibit, isig, itg = inner.comps[icid]
        k = -1
        if bit >= 0 or ibit >= 0:
            k = len(of_outer)
            of_outer.append(bit)
            of_inner.append(ibit)
        flips = sig ^ isig ^ outer.ins[b][2] ^ inner.virts[inner.outs[b][1][0][0]][2]
        comps.append([dim, k, bool(flips), list(itg)])
    if len(of_outer) > L.MAX_BITS:
        return None
    G.comps = comps
    codes = []
    for m in range(1 << len(of_outer)):
        x = outer.codes[sum(((m >> i) & 1) << o for i, o in enumerate(of_outer) if o >= 0)]
        y = inner.codes[sum(((m >> i) & 1) << o for i, o in enumerate(of_inner) if o >= 0)]
        codes.append(2 if 2 in (x, y) else x ^ y)
    G.set_table(codes)
    return G


def run_composed(outer, inner, src, dst=None, alpha=1.0):
    """outer(inner(src)) in one pass: `outer` is built against the contiguous tensor that `inner` would
    write.  One gather where the two compose (every contraction of a contraction), else gtn_permute2,
    which maps each element through both."""
    lib = L.lib()
    one = compose(outer, inner)
    if one is not None:
        return one.run(src, dst=dst, alpha=alpha)
    if dst is None:
        dst = DeviceArray.empty(outer.out_shape(), src.dtype)
    if dst.numel() == 0:
        return dst
    if not (src.is_contiguous() and dst.is_contiguous()):
        raise ValueError("gather operands must be contiguous")
    mid = 1
    for d in inner.out_shape():
        mid *= d
    do = outer.desc(L.dtype_code(src), mid, alpha)
    dn = inner.desc(L.dtype_code(src), src.numel())
    L.check(lib.gtn_permute2(C.byref(do), C.byref(dn), L.ptr(src), L.ptr(dst), L.stream_ptr()), "gtn_permute2")
    return dst


def strides(shape):
    st, acc = [0] * len(shape), 1
    for i in range(len(shape) - 1, -1, -1):
        st[i] = acc
        acc *= shape[i]
    return st


def source_axes(perm, shape, encs, sigmas=None, base_stride=None):
    """Register a plain C-ordered source tensor (one leg per axis); returns the input ids."""
    st = strides(shape) if base_stride is None else base_stride
    ids = []
    for a, dim in enumerate(shape):
        ids.append(perm.add_in(dim, st[a], enc=encs[a], sigma=(sigmas[a] if sigmas else False)))
    return ids
