// Integer index maps and sign factors on the device (param.py:61-83; __init__.py:1011-1154,
// 1944-2126, 2947-3170), and the FP64 reductions / elementwise helpers of the TRG step.
#include "gtn_common.h"
#include <stdlib.h>
#include <string.h>
#include <math.h>
#include <algorithm>
#include <vector>
#include <utility>
#include <map>
#include <mutex>
#include <shared_mutex>
#include <string>

namespace gtn {

static thread_local char g_err[1024] = "";
static std::vector<std::pair<uint64_t, uint64_t>> g_regions;
static bool g_dry = false;
bool dry_run() { return g_dry; }
int check_range(const void *p, int64_t bytes, const char *what) {
    if (!g_dry || bytes <= 0) return GTN_OK;
    uint64_t lo = (uint64_t)p, hi = lo + (uint64_t)bytes;
    for (auto &r : g_regions)
        if (r.first <= lo && hi <= r.first + r.second) return GTN_OK;
    set_error("dry run: %s touches [%#llx, %#llx) outside every registered region", what, (unsigned long long)lo,
              (unsigned long long)hi);
    return GTN_EINVAL;
}
void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

// ---------------------------------------------------------------------------------------------
// index tables
// ---------------------------------------------------------------------------------------------
__global__ void k_index_tables(int64_t n, int32_t *popc, int8_t *sigma, int32_t *enc) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        uint64_t u = (uint64_t)i;
        if (popc) popc[i] = (int32_t)popc64(u);
        if (sigma) sigma[i] = sigma_bit(u) ? (int8_t)-1 : (int8_t)1;
        if (enc) enc[i] = (int32_t)enc_switch(u);
    }
}

// ---------------------------------------------------------------------------------------------
// signed gather.  The descriptor lives in kernel-argument memory, so every lane reads the same
// words.  Division by an axis dimension is a shift when the dimension is a power of two (all
// fermionic legs are) and a true division otherwise.
// ---------------------------------------------------------------------------------------------
constexpr int AX = GTN_PERM_MAX_AX, NC = GTN_PERM_MAX_COMP;
struct PermArgs {
    int32_t n_out, n_virt, n_comp, n_in;
    int32_t virt_enc_mask, virt_sigma_mask, comp_sigma_mask, in_enc_mask, in_sigma_mask, in_split_mask;
    uint32_t out_dim[AX];
    int8_t out_shift[AX];
    int8_t out_virt[AX][2];
    int64_t out_vmul[AX][2];
    int8_t virt_ncomp[AX];
    uint32_t comp_dim[NC];
    int8_t comp_shift[NC];
    int8_t comp_bit[NC];
    int8_t comp_in[NC][2];
    int64_t comp_mult[NC][2];
    int64_t in_stride[AX];
    int64_t in_stride_lo[AX];
    uint32_t table[2 * (1 << GTN_PERM_MAX_BITS) / 32];
    double alpha_re, alpha_im;
    int64_t total;
};

// Contribution of the virtual axes in `vmask` for virtual-axis values V: their components' parity
// bits and sign flips, and the offset and sign flips of the input axes in `inmask`.  With every
// axis in the masks this is the whole map; a subset is exact when the inputs in `inmask` are fed
// only by components of the virtual axes in `vmask` (inputs fed by nobody hold index 0, whose
// offset, encoding and sigma are all trivial).
__device__ __forceinline__ void perm_core(const PermArgs &a, const uint64_t (&V)[AX], uint32_t vmask,
                                          uint32_t inmask, int64_t &off, uint32_t &bits, uint32_t &neg) {
    uint64_t F[AX];
#pragma unroll
    for (int b = 0; b < AX; ++b) F[b] = 0;
    bits = 0;
    neg = 0;
    int j = a.n_comp;
    for (int v = a.n_virt - 1; v >= 0; --v) {
        if (!((vmask >> v) & 1u)) {
            j -= a.virt_ncomp[v];
            continue;
        }
        uint64_t c = ((a.virt_enc_mask >> v) & 1) ? enc_switch(V[v]) : V[v];
        if ((a.virt_sigma_mask >> v) & 1) neg ^= sigma_bit(c);
        for (int t = 0; t < a.virt_ncomp[v]; ++t) {
            --j;
            uint64_t d = a.comp_dim[j], k;
            if (a.comp_shift[j] >= 0) {
                k = c & (d - 1);
                c >>= a.comp_shift[j];
            } else {
                k = c % d;
                c /= d;
            }
            uint32_t pc = popc64(k);
            if (a.comp_bit[j] >= 0) bits ^= (pc & 1u) << a.comp_bit[j];
            if ((a.comp_sigma_mask >> j) & 1) neg ^= (pc >> 1) & 1u;
            F[a.comp_in[j][0]] += k * (uint64_t)a.comp_mult[j][0];
            if (a.comp_in[j][1] >= 0) F[a.comp_in[j][1]] += k * (uint64_t)a.comp_mult[j][1];
        }
    }
    off = 0;
    for (int b = 0; b < a.n_in; ++b) {
        if (!((inmask >> b) & 1u)) continue;
        uint64_t f = F[b];
        if ((a.in_sigma_mask >> b) & 1) neg ^= sigma_bit(f);
        uint64_t e = ((a.in_enc_mask >> b) & 1) ? enc_switch(f) : f;
        if ((a.in_split_mask >> b) & 1)
            off += (int64_t)(e & 1) * a.in_stride_lo[b] + (int64_t)(e >> 1) * a.in_stride[b];
        else
            off += (int64_t)e * a.in_stride[b];
    }
}

__device__ __forceinline__ uint32_t sign_code(const PermArgs &a, uint32_t bits, uint32_t neg) {
    uint32_t t = (a.table[bits >> 4] >> ((bits & 15u) * 2)) & 3u;
    return (t == 2u) ? 2u : (t ^ neg);
}

// Returns the source offset of output element `lin` and its table entry (0: +1, 1: -1, 2: zero).
__device__ __forceinline__ int64_t perm_map(const PermArgs &a, uint64_t lin, uint32_t &code) {
    uint64_t V[AX];
#pragma unroll
    for (int b = 0; b < AX; ++b) V[b] = 0;
    uint64_t rest = lin;
    for (int ax = a.n_out - 1; ax >= 0; --ax) {
        uint64_t d = a.out_dim[ax], o;
        if (a.out_shift[ax] >= 0) {
            o = rest & (d - 1);
            rest >>= a.out_shift[ax];
        } else {
            o = rest % d;
            rest /= d;
        }
        if (a.out_virt[ax][0] >= 0) V[a.out_virt[ax][0]] += o * (uint64_t)a.out_vmul[ax][0];
        if (a.out_virt[ax][1] >= 0) V[a.out_virt[ax][1]] += o * (uint64_t)a.out_vmul[ax][1];
    }
    int64_t off;
    uint32_t bits, neg;
    perm_core(a, V, 0xffffffffu, 0xffffffffu, off, bits, neg);
    code = sign_code(a, bits, neg);
    return off;
}

// ---------------------------------------------------------------------------------------------
// Table-driven map.  The virtual axes fall into groups: two virtual axes share a group when their
// components feed a common input axis.  A group's contribution (source offset, parity bits, sign
// flip) depends only on the values of its own virtual axes, so it is tabulated once per gather
// shape, indexed by G = the mixed-radix number of the output indices that feed those axes, in an order
// that keeps the lanes of a wavefront on consecutive entries.  Where every extent and stride is a power of two and no two indices share bits of the
// offset, the map is linear over GF(2) (the encoder, the split and the parities are exclusive ors of the
// index bits), so every virtual axis is a group of its own and the groups' offsets combine by exclusive
// or, whatever input axes they share: the operand gather of a contraction's output, whose fused GEMM
// indices mix the legs of both operand groups, has tables of a few thousand entries instead of none.  Per element the map is then an index decomposition, at most kTabGroups table
// reads, a sum and an XOR, instead of the component walk of perm_map.
// ---------------------------------------------------------------------------------------------
constexpr int kTabGroups = 4;
// source offset in the low 53 bits, parity bits from bit 53, sign flip in bit 63
typedef uint64_t TabEntry;
constexpr int kTabOffBits = 53;
constexpr uint32_t kTabNeg = 1u << (63 - kTabOffBits);
struct TabArgs {
    int32_t ng;
    uint32_t gmul[AX][kTabGroups];  // G_g = sum_ax o_ax * gmul[ax][g]
    const TabEntry *tab[kTabGroups];
    uint64_t signs;   // the sign table's first 32 entries, and whether it has no more
    int32_t short_signs;
    int32_t lin;      // offsets combine by exclusive or, else by addition
};
struct TabBuild {
    int32_t ng;
    int64_t start[kTabGroups + 1];  // first entry of each group's table
    uint32_t vmask[kTabGroups], inmask[kTabGroups];
    int32_t nx[kTabGroups];  // the output axes that feed the group and their radices in its table
    int8_t ax[kTabGroups][AX];
    uint32_t rad[kTabGroups][AX];
};

__global__ void k_perm_tables(PermArgs a, TabBuild t, TabEntry *out) {
    const int64_t n = t.start[t.ng];
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        int g = 0;
        while (g + 1 < t.ng && e >= t.start[g + 1]) ++g;
        const uint32_t G = (uint32_t)(e - t.start[g]);
        uint64_t V[AX];
#pragma unroll
        for (int b = 0; b < AX; ++b) V[b] = 0;
        for (int i = 0; i < t.nx[g]; ++i) {
            const int ax = t.ax[g][i];
            const uint64_t o = (G / t.rad[g][i]) % a.out_dim[ax];
            if (a.out_virt[ax][0] >= 0) V[a.out_virt[ax][0]] += o * (uint64_t)a.out_vmul[ax][0];
            if (a.out_virt[ax][1] >= 0) V[a.out_virt[ax][1]] += o * (uint64_t)a.out_vmul[ax][1];
        }
        int64_t off;
        uint32_t bits, neg;
        perm_core(a, V, t.vmask[g], t.inmask[g], off, bits, neg);
        out[e] = (uint64_t)off | ((uint64_t)(bits | (neg ? kTabNeg : 0u)) << kTabOffBits);
    }
}

__device__ __forceinline__ int64_t tab_join(const TabArgs &t, int64_t x, int64_t y) { return t.lin ? x ^ y : x + y; }
// adds a table entry to an offset and a code (parity bits and sign flip)
__device__ __forceinline__ void tab_add(const TabArgs &t, TabEntry e, int64_t &off, uint32_t &c) {
    off = tab_join(t, off, (int64_t)(e & (((uint64_t)1 << kTabOffBits) - 1)));
    c ^= (uint32_t)(e >> kTabOffBits);
}
// sign table entry (0: +1, 1: -1, 2: zero) of a code; tables of up to five parity bits sit in a register
__device__ __forceinline__ uint32_t tab_sign(const PermArgs &a, const TabArgs &t, uint32_t c) {
    const uint32_t bits = c & (kTabNeg - 1);
    if (!t.short_signs) return sign_code(a, bits, c / kTabNeg);
    const uint32_t s = (uint32_t)(t.signs >> (2 * bits)) & 3u;
    return s == 2u ? 2u : (s ^ (c / kTabNeg));
}

// Table indices of the output axes 0 .. hi for the row-major index `lin` over those axes.
__device__ __forceinline__ void tab_index(const PermArgs &a, const TabArgs &t, uint64_t lin, int hi,
                                          uint32_t (&G)[kTabGroups]) {
#pragma unroll
    for (int g = 0; g < kTabGroups; ++g) G[g] = 0;
    uint64_t rest = lin;
    for (int ax = hi; ax >= 0; --ax) {
        uint32_t o;
        if (a.out_shift[ax] >= 0) {
            o = (uint32_t)(rest & (uint64_t)(a.out_dim[ax] - 1));
            rest >>= a.out_shift[ax];
        } else if ((rest >> 32) == 0) {
            const uint32_t r32 = (uint32_t)rest, d = a.out_dim[ax];
            o = r32 % d;
            rest = r32 / d;
        } else {
            o = (uint32_t)(rest % a.out_dim[ax]);
            rest /= a.out_dim[ax];
        }
#pragma unroll
        for (int g = 0; g < kTabGroups; ++g) G[g] += o * t.gmul[ax][g];
    }
}

__device__ __forceinline__ int64_t tab_map(const PermArgs &a, const TabArgs &t, uint64_t lin, uint32_t &code) {
    uint32_t G[kTabGroups];
    tab_index(a, t, lin, a.n_out - 1, G);
    int64_t off = 0;
    uint32_t c = 0;
#pragma unroll
    for (int g = 0; g < kTabGroups; ++g)
        if (g < t.ng) tab_add(t, t.tab[g][G[g]], off, c);
    code = tab_sign(a, t, c);
    return off;
}

template <bool TAB>
__device__ __forceinline__ int64_t map_elem(const PermArgs &a, const TabArgs &t, uint64_t lin, uint32_t &code) {
    if constexpr (TAB)
        return tab_map(a, t, lin, code);
    else
        return perm_map(a, lin, code);
}

// A workgroup takes kPermUnroll * 256 consecutive output elements per pass, a lane every 256th of
// them (each load instruction stays coalesced, and the workgroups sweep the output in order, which
// keeps the source lines they share in L2); a lane issues the index maps and table reads of its
// kPermUnroll elements together, then their source reads, so kPermUnroll dependent load chains are in
// flight per lane instead of one.
constexpr int kPermUnroll = 4;

template <typename T, bool TAB>
__global__ void __launch_bounds__(256) k_permute(PermArgs a, TabArgs tb, const T *__restrict__ src, T *__restrict__ dst) {
    const double al = a.alpha_re;
    const int64_t chunk = (int64_t)kPermUnroll * blockDim.x;
    for (int64_t i0 = blockIdx.x * chunk + threadIdx.x; i0 < a.total; i0 += (int64_t)gridDim.x * chunk) {
        int64_t off[kPermUnroll];
        uint32_t code[kPermUnroll];
#pragma unroll
        for (int u = 0; u < kPermUnroll; ++u) {
            const int64_t i = i0 + u * (int64_t)blockDim.x;
            code[u] = 2u;
            off[u] = 0;
            if (i < a.total) off[u] = map_elem<TAB>(a, tb, (uint64_t)i, code[u]);
        }
        double v[kPermUnroll];
#pragma unroll
        for (int u = 0; u < kPermUnroll; ++u) v[u] = (code[u] == 2u) ? 0.0 : (double)src[off[u]];
#pragma unroll
        for (int u = 0; u < kPermUnroll; ++u) {
            const int64_t i = i0 + u * (int64_t)blockDim.x;
            if (i < a.total) dst[i] = (T)(code[u] == 2u ? 0.0 : v[u] * (code[u] ? -al : al));
        }
    }
}

// Row walk of a table-driven gather.  The output is rows of `width` consecutive elements, the trailing
// ns axes; a workgroup takes one chunk of U * 256 columns of `rows_per` rows, one after another.  What
// the leading axes add to the table indices is the same in every lane: groups that no trailing axis
// feeds are looked up once per row, the others (usually one) per element, and not again while their
// leading part stays the same.  An element then costs a source read and a few integer operations where
// the walk above reads up to four entries for it.  MI355X, 64^4 doubles: encoder switch 71 -> 52 us
// (5.2 TB/s), operand gathers of a contraction 55 -> 44 us (6.1 TB/s); tiles (below) with the same
// economy 164 -> 82 us; 8^4 doubles 20 -> 5 us.
struct RowArgs {
    int64_t width, rows;
    int32_t ns, chunks, rows_per;
    uint32_t vary;  // groups that the trailing axes feed
};
template <typename T, int U>
__global__ void __launch_bounds__(256) k_permute_rows(PermArgs a, TabArgs tb, RowArgs w, const T *__restrict__ src,
                                                      T *__restrict__ dst) {
    const double al = a.alpha_re;
    const int last = a.n_out - 1, lead = last - w.ns;
    const int64_t c0 = (int64_t)(blockIdx.x % w.chunks) * (U * 256);
    const int64_t r0 = (int64_t)(blockIdx.x / w.chunks) * w.rows_per;
    const int64_t r1 = r0 + w.rows_per < w.rows ? r0 + w.rows_per : w.rows;
    // table indices of this lane's columns
    uint32_t Gc[U][kTabGroups];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int g = 0; g < kTabGroups; ++g) Gc[u][g] = 0;
        uint32_t c = (uint32_t)c0 + threadIdx.x + u * 256;
        for (int ax = last; ax > lead; --ax) {
            uint32_t o = c;
            if (ax > lead + 1 && a.out_shift[ax] >= 0) {
                o = c & (a.out_dim[ax] - 1);
                c >>= a.out_shift[ax];
            } else if (ax > lead + 1) {  // once a lane and column, for all rows
                o = c % a.out_dim[ax];
                c /= a.out_dim[ax];
            }
#pragma unroll
            for (int g = 0; g < kTabGroups; ++g) Gc[u][g] += o * tb.gmul[ax][g];
        }
    }
    int64_t offc[U];
    uint32_t cc[U];
    uint32_t Gv[kTabGroups];  // the leading part of the varying groups that offc and cc hold
    for (int64_t row = r0; row < r1; ++row) {
        uint32_t G[kTabGroups];
        tab_index(a, tb, (uint64_t)row, lead, G);
        int64_t offr = 0;
        uint32_t cr = 0;
        bool same = row > r0;
#pragma unroll
        for (int g = 0; g < kTabGroups; ++g)
            if (g < tb.ng) {
                if ((w.vary >> g) & 1u) {
                    same = same && G[g] == Gv[g];
                    Gv[g] = G[g];
                } else {
                    tab_add(tb, tb.tab[g][G[g]], offr, cr);
                }
            }
        if (!same) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                offc[u] = 0;
                cc[u] = 0;
            }
#pragma unroll
            for (int g = 0; g < kTabGroups; ++g)
                if (g < tb.ng && ((w.vary >> g) & 1u)) {
#pragma unroll
                    for (int u = 0; u < U; ++u) tab_add(tb, tb.tab[g][G[g] + Gc[u][g]], offc[u], cc[u]);
                }
        }
        uint32_t code[U];
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            code[u] = tab_sign(a, tb, cc[u] ^ cr);
            v[u] = code[u] == 2u ? 0.0 : (double)src[tab_join(tb, offc[u], offr)];
        }
        T *d = dst + row * w.width + c0 + threadIdx.x;
#pragma unroll
        for (int u = 0; u < U; ++u) d[u * 256] = (T)(code[u] == 2u ? 0.0 : v[u] * (code[u] ? -al : al));
    }
}

// Two gathers in one pass: dst[i] = sign_o(i) sign_n(j) src[off_n(j)] with j = off_o(i), the outer
// gather's source offset, read as the inner gather's output index (the inner gather's output is the
// contiguous tensor the outer one would have read).  Same lane arrangement as k_permute.
template <typename T, bool TABO, bool TABN>
__global__ void __launch_bounds__(256) k_permute2(PermArgs ao, TabArgs to, PermArgs an, TabArgs tn,
                                                  const T *__restrict__ src, T *__restrict__ dst) {
    const double al = ao.alpha_re * an.alpha_re;
    const int64_t chunk = (int64_t)kPermUnroll * blockDim.x;
    for (int64_t i0 = blockIdx.x * chunk + threadIdx.x; i0 < ao.total; i0 += (int64_t)gridDim.x * chunk) {
        int64_t off[kPermUnroll];
        uint32_t code[kPermUnroll];
#pragma unroll
        for (int u = 0; u < kPermUnroll; ++u) {
            const int64_t i = i0 + u * (int64_t)blockDim.x;
            code[u] = 2u;
            off[u] = 0;
            if (i < ao.total) {
                uint32_t co, cn;
                const int64_t j = map_elem<TABO>(ao, to, (uint64_t)i, co);
                if (co != 2u) {
                    off[u] = map_elem<TABN>(an, tn, (uint64_t)j, cn);
                    code[u] = cn == 2u ? 2u : (co ^ cn);
                }
            }
        }
        double v[kPermUnroll];
#pragma unroll
        for (int u = 0; u < kPermUnroll; ++u) v[u] = (code[u] == 2u) ? 0.0 : (double)src[off[u]];
#pragma unroll
        for (int u = 0; u < kPermUnroll; ++u) {
            const int64_t i = i0 + u * (int64_t)blockDim.x;
            if (i < ao.total) dst[i] = (T)(code[u] == 2u ? 0.0 : v[u] * (code[u] ? -al : al));
        }
    }
}

__global__ void k_permute_c128(PermArgs a, const double2 *__restrict__ src, double2 *__restrict__ dst) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.total; i += (int64_t)gridDim.x * blockDim.x) {
        uint32_t code;
        int64_t off = perm_map(a, (uint64_t)i, code);
        double2 r = {0.0, 0.0};
        if (code != 2u) {
            double2 v = src[off];
            double s = code ? -1.0 : 1.0;
            r.x = s * (a.alpha_re * v.x - a.alpha_im * v.y);
            r.y = s * (a.alpha_re * v.y + a.alpha_im * v.x);
        }
        dst[i] = r;
    }
}

// Workgroups of a gather at most (about: HIP refuses 2^32 work items in a dimension, 2^24 workgroups of 256)
constexpr int64_t kMaxGrid = 1 << 23;

// Tiled variant for gathers whose output's last axis is far apart in the source: output axis t1
// (the one whose consecutive indices share the most source lines) and the last output axis t0 form
// n1 x n0 tiles.  A tile is read with t1 fastest (consecutive source addresses), staged in LDS with its
// signs applied, and written with t0 fastest (consecutive output addresses).  Fused output axes are cut
// into their legs first (split_axes): the leg that runs through consecutive addresses is often the upper
// part of a fused index.  MI355X, eight 64^4 tensors: joins into parity blocks 738 -> 557 us, operand
// gathers of the largest contraction 827 -> 478 us (the row walk before).
struct TileArgs {
    int32_t t0, t1, n_rest, tiles0, tiles1;
    int32_t sh0, sh1;  // n0 = 1 << sh0, n1 = 1 << sh1: 16, 32 or 64
    uint32_t slot0;    // first tile of each XCD's share that this launch does
    int32_t rest_ax[AX];
    int64_t ostr[AX];
    int64_t rest_total;
};

template <typename T, bool TAB>
__global__ void __launch_bounds__(256) k_permute_tiled(PermArgs a, TabArgs tb, TileArgs t, const T *__restrict__ src,
                                                       T *__restrict__ dst) {
    HIP_DYNAMIC_SHARED(double, tile)  // n1 x (n0 + 1)
    const double al = a.alpha_re;
    const uint32_t per = (uint32_t)t.tiles0 * t.tiles1;
    const int d1 = (int)a.out_dim[t.t1], d0 = (int)a.out_dim[t.t0];
    const int64_t s1 = t.ostr[t.t1];
    const int n0 = 1 << t.sh0, n1 = 1 << t.sh1, ld = n0 + 1, count = n0 << t.sh1;
    // element e = tid + 256 u of a tile: l1 = e % n1 (the same for every u), l0 = e / n1
    const int l1 = threadIdx.x & (n1 - 1), l0s = threadIdx.x >> t.sh1, l0d = 256 >> t.sh1;
    // one tile per workgroup, the tiles of an XCD consecutive (its L2 has the lines that neighbours share)
    const uint32_t nblk = per * (uint32_t)t.rest_total, share = (nblk + 7) / 8, slot = t.slot0 + (blockIdx.x >> 3);
    const uint32_t blk = (blockIdx.x & 7) * share + slot;
    if (blk < nblk && slot < share) {
        uint32_t rr = per == 1 ? blk : blk / per;
        const uint32_t q = blk - rr * per;
        const int i1b = (int)(per == 1 ? 0 : q / (uint32_t)t.tiles0) << t.sh1;
        const int i0b = (int)(per == 1 ? 0 : q % (uint32_t)t.tiles0) << t.sh0;
        int64_t base = 0;
        uint32_t Gb[kTabGroups];
        if constexpr (TAB) {
#pragma unroll
            for (int g = 0; g < kTabGroups; ++g)
                Gb[g] = (uint32_t)i1b * tb.gmul[t.t1][g] + (uint32_t)i0b * tb.gmul[t.t0][g];
        }
        for (int k = t.n_rest - 1; k >= 0; --k) {
            const int ax = t.rest_ax[k];
            uint32_t o;
            if (a.out_shift[ax] >= 0) {
                o = rr & (a.out_dim[ax] - 1);
                rr >>= a.out_shift[ax];
            } else {
                o = rr % a.out_dim[ax];
                rr /= a.out_dim[ax];
            }
            base += o * t.ostr[ax];
            if constexpr (TAB) {
#pragma unroll
                for (int g = 0; g < kTabGroups; ++g) Gb[g] += o * tb.gmul[ax][g];
            }
        }
        // with tables, groups that t0 does not feed are looked up once per lane
        const bool in1 = i1b + l1 < d1;
        int64_t off1 = 0;
        uint32_t c1 = 0;
        if constexpr (TAB) {
#pragma unroll
            for (int g = 0; g < kTabGroups; ++g)
                if (g < tb.ng && tb.gmul[t.t0][g] == 0)
                    tab_add(tb, tb.tab[g][Gb[g] + (in1 ? (uint32_t)l1 * tb.gmul[t.t1][g] : 0u)], off1, c1);
        }
        // up to 16 elements per lane in batches of 8: index maps and table reads first, then the source
        // reads, so that 8 load chains are in flight per lane
        for (int e0 = 0; e0 < count; e0 += 8 * 256) {
            int64_t off[8];
            uint32_t code[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int l0 = l0s + ((e0 >> 8) + u) * l0d;
                const int i0 = i0b + l0;
                code[u] = 2u;
                off[u] = 0;
                if (in1 && l0 < n0 && i0 < d0) {
                    if constexpr (TAB) {
                        uint32_t c = c1;
                        off[u] = off1;
#pragma unroll
                        for (int g = 0; g < kTabGroups; ++g)
                            if (g < tb.ng && tb.gmul[t.t0][g] != 0)
                                tab_add(tb, tb.tab[g][Gb[g] + (uint32_t)l0 * tb.gmul[t.t0][g] + (uint32_t)l1 * tb.gmul[t.t1][g]],
                                        off[u], c);
                        code[u] = tab_sign(a, tb, c);
                    } else {
                        off[u] = map_elem<TAB>(a, tb, (uint64_t)(base + (i1b + l1) * s1 + i0), code[u]);
                    }
                }
            }
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = (code[u] == 2u) ? 0.0 : (double)src[off[u]] * (code[u] ? -al : al);
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int l0 = l0s + ((e0 >> 8) + u) * l0d;
                if (l0 < n0) tile[l1 * ld + l0] = v[u];
            }
        }
        __syncthreads();
        for (int e = threadIdx.x; e < count; e += 256) {
            const int w0 = e & (n0 - 1), w1 = e >> t.sh0;
            const int i1 = i1b + w1, i0 = i0b + w0;
            if (i1 < d1 && i0 < d0) dst[base + i1 * s1 + i0] = (T)tile[w1 * ld + w0];
        }
    }
}

static int ilog2_exact(uint64_t d) {
    if (d == 0 || (d & (d - 1))) return -1;
    int s = 0;
    while ((1ull << s) < d) ++s;
    return s;
}

static int build_perm_args(const gtn_perm_desc *d, PermArgs &a) {
    GTN_REQUIRE(d->n_out >= 0 && d->n_out <= AX, "gtn_permute: n_out out of range");
    GTN_REQUIRE(d->n_virt >= 0 && d->n_virt <= AX, "gtn_permute: n_virt out of range");
    GTN_REQUIRE(d->n_comp >= 0 && d->n_comp <= NC, "gtn_permute: n_comp out of range");
    GTN_REQUIRE(d->n_in >= 0 && d->n_in <= AX, "gtn_permute: n_in out of range");
    GTN_REQUIRE(d->n_bits >= 0 && d->n_bits <= GTN_PERM_MAX_BITS, "gtn_permute: n_bits out of range");
    memset(&a, 0, sizeof(a));
    a.n_out = d->n_out;
    a.n_virt = d->n_virt;
    a.n_comp = d->n_comp;
    a.n_in = d->n_in;
    int64_t total = 1;
    int64_t vmax[AX] = {0};
    for (int ax = 0; ax < d->n_out; ++ax) {
        GTN_REQUIRE(d->out_dim[ax] >= 0 && d->out_dim[ax] < (1ll << 31), "gtn_permute: bad out_dim");
        total *= d->out_dim[ax];
        a.out_dim[ax] = (uint32_t)d->out_dim[ax];
        a.out_shift[ax] = (int8_t)ilog2_exact((uint64_t)d->out_dim[ax]);
        for (int t = 0; t < 2; ++t) {
            int v = d->out_virt[ax][t];
            GTN_REQUIRE(v >= -1 && v < d->n_virt, "gtn_permute: out_virt out of range");
            GTN_REQUIRE(d->out_vmul[ax][t] >= 0, "gtn_permute: negative out_vmul");
            a.out_virt[ax][t] = (int8_t)v;
            a.out_vmul[ax][t] = d->out_vmul[ax][t];
            if (v >= 0 && d->out_dim[ax] > 0) vmax[v] += (d->out_dim[ax] - 1) * d->out_vmul[ax][t];
        }
    }
    int jc = 0;
    int64_t fmax[AX] = {0};
    for (int v = 0; v < d->n_virt; ++v) {
        GTN_REQUIRE(d->virt_dim[v] >= 1, "gtn_permute: bad virt_dim");
        GTN_REQUIRE(vmax[v] < d->virt_dim[v], "gtn_permute: virtual axis %d overflows", v);
        if (d->virt_enc[v]) {
            // eps only flips the lowest bit, so it maps [0, d) onto itself for every even d (a fused
            // index of fermionic and bosonic legs is even but need not be a power of two)
            GTN_REQUIRE(d->virt_dim[v] % 2 == 0 || d->virt_dim[v] == 1, "gtn_permute: encoder on an odd axis");
            a.virt_enc_mask |= 1 << v;
        }
        if (d->virt_sigma[v]) a.virt_sigma_mask |= 1 << v;
        a.virt_ncomp[v] = (int8_t)d->virt_ncomp[v];
        int64_t prod = 1;
        for (int t = 0; t < d->virt_ncomp[v]; ++t, ++jc) {
            GTN_REQUIRE(jc < d->n_comp, "gtn_permute: components do not add up");
            prod *= d->comp_dim[jc];
        }
        GTN_REQUIRE(prod == d->virt_dim[v], "gtn_permute: components of virtual axis %d do not multiply to its dim", v);
    }
    GTN_REQUIRE(jc == d->n_comp, "gtn_permute: components do not add up");
    for (int j = 0; j < d->n_comp; ++j) {
        GTN_REQUIRE(d->comp_dim[j] >= 1 && d->comp_dim[j] < (1ll << 31), "gtn_permute: bad comp_dim");
        a.comp_dim[j] = (uint32_t)d->comp_dim[j];
        a.comp_shift[j] = (int8_t)ilog2_exact((uint64_t)d->comp_dim[j]);
        GTN_REQUIRE(d->comp_bit[j] >= -1 && d->comp_bit[j] < d->n_bits, "gtn_permute: comp_bit beyond n_bits");
        a.comp_bit[j] = (int8_t)d->comp_bit[j];
        if (d->comp_sigma[j]) a.comp_sigma_mask |= 1 << j;
        GTN_REQUIRE(d->comp_in[j][0] >= 0 && d->comp_in[j][0] < d->n_in, "gtn_permute: comp_in out of range");
        GTN_REQUIRE(d->comp_in[j][1] >= -1 && d->comp_in[j][1] < d->n_in, "gtn_permute: comp_in out of range");
        for (int t = 0; t < 2; ++t) {
            a.comp_in[j][t] = (int8_t)d->comp_in[j][t];
            a.comp_mult[j][t] = d->comp_mult[j][t];
            GTN_REQUIRE(d->comp_mult[j][t] >= 0, "gtn_permute: negative comp_mult");
            if (d->comp_in[j][t] >= 0) fmax[d->comp_in[j][t]] += (d->comp_dim[j] - 1) * d->comp_mult[j][t];
        }
    }
    // bounds: every fused input index stays inside its axis, the furthest element inside src
    int64_t far = 0;
    for (int b = 0; b < d->n_in; ++b) {
        GTN_REQUIRE(fmax[b] < d->in_dim[b], "gtn_permute: input axis %d overflows (%lld >= %lld)", b, (long long)fmax[b],
                    (long long)d->in_dim[b]);
        if (d->in_enc[b]) {
            GTN_REQUIRE(d->in_dim[b] % 2 == 0 || d->in_dim[b] == 1, "gtn_permute: encoder on an odd input axis");
            a.in_enc_mask |= 1 << b;
        }
        if (d->in_sigma[b]) a.in_sigma_mask |= 1 << b;
        GTN_REQUIRE(d->in_stride[b] >= 0 && d->in_stride_lo[b] >= 0, "gtn_permute: negative stride");
        a.in_stride[b] = d->in_stride[b];
        a.in_stride_lo[b] = d->in_stride_lo[b];
        // the largest encoded index is in_dim - 1 (eps maps [0, d) onto itself for even d)
        int64_t emax = d->in_dim[b] - 1;
        if (d->in_split[b]) {
            a.in_split_mask |= 1 << b;
            GTN_REQUIRE(d->in_dim[b] % 2 == 0 || d->in_dim[b] == 1, "gtn_permute: split axis needs an even dim");
            far += (emax >= 1 ? d->in_stride_lo[b] : 0) + (emax >> 1) * d->in_stride[b];
        } else {
            far += emax * d->in_stride[b];
        }
    }
    GTN_REQUIRE(total == 0 || far < d->src_elems, "gtn_permute: source too small (%lld needed, %lld given)",
                (long long)far + 1, (long long)d->src_elems);
    memcpy(a.table, d->table, sizeof(a.table));
    a.alpha_re = d->alpha_re;
    a.alpha_im = d->alpha_im;
    a.total = total;
    return GTN_OK;
}

// ---------------------------------------------------------------------------------------------
// sign tensor (diagnostic output of the reference's S1 / S3)
// ---------------------------------------------------------------------------------------------
struct SignArgs {
    int32_t ndim;
    uint32_t dims[GTN_PERM_MAX_BITS];
    uint32_t table[(1 << GTN_PERM_MAX_BITS) / 32];
    int64_t total;
};

__global__ void k_sign_tensor(SignArgs a, int8_t *out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.total; i += (int64_t)gridDim.x * blockDim.x) {
        uint64_t r = (uint64_t)i;
        uint32_t bits = 0;
        for (int ax = a.ndim - 1; ax >= 0; --ax) {
            uint64_t k = r % a.dims[ax];
            r /= a.dims[ax];
            bits |= (popc64(k) & 1u) << ax;
        }
        out[i] = ((a.table[bits >> 5] >> (bits & 31u)) & 1u) ? (int8_t)-1 : (int8_t)1;
    }
}

// ---------------------------------------------------------------------------------------------
// reductions (FP64 accumulation, deterministic two-pass: per-block partials then one block)
// ---------------------------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ double sq(T v) { return (double)v * (double)v; }
template <>
__device__ __forceinline__ double sq<double2>(double2 v) { return v.x * v.x + v.y * v.y; }

__device__ __forceinline__ double block_sum(double v, double *sh) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0) {
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) t += sh[i];
    }
    __syncthreads();
    return t;
}

template <typename T>
__global__ void k_sumsq_partial(const T *__restrict__ x, int64_t n, double *part) {
    __shared__ double sh[16];
    double acc = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        acc += sq(x[i]);
    double t = block_sum(acc, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

__global__ void k_sum_final(const double *part, int np, double *out) {
    __shared__ double sh[16];
    double acc = 0;
    for (int i = threadIdx.x; i < np; i += blockDim.x) acc += part[i];
    double t = block_sum(acc, sh);
    if (threadIdx.x == 0) out[0] = t;
}

template <typename T>
__global__ void k_scale_by_norm(T *x, int64_t n, const double *nrm2) {
    double inv = 1.0 / sqrt(nrm2[0]);
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = (T)((double)x[i] * inv);
}
__global__ void k_scale_by_norm_c(double2 *x, int64_t n, const double *nrm2) {
    double inv = 1.0 / sqrt(nrm2[0]);
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double2 v = x[i];
        v.x *= inv;
        v.y *= inv;
        x[i] = v;
    }
}

template <typename T>
__global__ void k_reduce_last(const T *__restrict__ src, T *__restrict__ dst, int64_t rows, int64_t inner) {
    for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < rows; r += (int64_t)gridDim.x * blockDim.x) {
        double acc = 0;
        for (int64_t t = 0; t < inner; ++t) acc += (double)src[r * inner + t];
        dst[r] = (T)acc;
    }
}
__global__ void k_reduce_last_c(const double2 *__restrict__ src, double2 *__restrict__ dst, int64_t rows, int64_t inner) {
    for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < rows; r += (int64_t)gridDim.x * blockDim.x) {
        double2 acc = {0, 0};
        for (int64_t t = 0; t < inner; ++t) {
            acc.x += src[r * inner + t].x;
            acc.y += src[r * inner + t].y;
        }
        dst[r] = acc;
    }
}

__global__ void k_lognorm(double *ln, const double *nrm2) {
    if (threadIdx.x == 0 && blockIdx.x == 0) ln[0] = 2.0 * ln[0] + 0.5 * log(nrm2[0]);
}

// ---- batched normalisation: every point b of a batch of nb tensors (n elements each) --------------
// pass 1: per-point partial sums of squares, grid (G, nb); part[b * G + g]
template <typename T>
__global__ void k_sumsq_batch_partial(const T *__restrict__ x, int64_t n, double *part) {
    __shared__ double sh[16];
    const T *xb = x + (int64_t)blockIdx.y * n;
    double acc = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        acc += sq(xb[i]);
    double t = block_sum(acc, sh);
    if (threadIdx.x == 0) part[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = t;
}
// pass 2, one workgroup per point: nrm2[b]; the driver's log-norm rule (example.py:192)
// lognorm[b] = 2 lognorm[b] + log ||T_b||; hist[b * hist_len + step] = log ||T_b|| while step < hist_len
__global__ void k_norm_batch_final(const double *part, int G, double *nrm2, double *lognorm, double *hist,
                                   int hist_len, const double *step) {
    __shared__ double sh[16];
    const int b = blockIdx.x;
    double acc = 0;
    for (int i = threadIdx.x; i < G; i += blockDim.x) acc += part[(int64_t)b * G + i];
    double t = block_sum(acc, sh);
    if (threadIdx.x == 0) {
        nrm2[b] = t;
        const double ln = 0.5 * log(t);
        if (lognorm) lognorm[b] = 2.0 * lognorm[b] + ln;
        if (hist && step) {
            const int k = (int)step[0];
            if (k >= 0 && k < hist_len) hist[(int64_t)b * hist_len + k] = ln;
        }
    }
}
// pass 3: x_b /= ||x_b||, grid (G, nb)
template <typename T>
__global__ void k_scale_batch(const T *x, T *dst, int64_t n, const double *nrm2) {
    const double inv = 1.0 / sqrt(nrm2[blockIdx.y]);
    const T *xb = x + (int64_t)blockIdx.y * n;
    T *db = dst + (int64_t)blockIdx.y * n;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        db[i] = (T)((double)xb[i] * inv);
}
__global__ void k_step_increment(double *step) {
    if (threadIdx.x == 0 && blockIdx.x == 0) step[0] += 1.0;
}
// dst (nb, 2d, 2d) = diagonal matrices whose entry (r, r) is src[b][r % 2][r / 2] (src (nb, 2, d)):
// the singular values of the even and odd parity blocks interleaved by the parity-preserving index
template <typename T>
__global__ void k_diag_interleave(T *dst, int64_t nb, int64_t d, const T *src) {
    const int64_t w = 2 * d, total = nb * w * w;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = e / (w * w), rc = e - b * w * w, r = rc / w, c = rc - r * w;
        dst[e] = (r == c) ? src[b * w + (r & 1) * d + (r >> 1)] : (T)0;
    }
}

template <typename T>
__global__ void k_power_diag(T *x, int64_t n, int64_t stride, double p, double rcond) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double v = (double)x[i * stride];
        x[i * stride] = (T)(fabs(v) > rcond ? pow(v, p) : 0.0);
    }
}

template <typename T>
__global__ void k_elementwise(T *x, int64_t n, int op, double p, double rcond) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const double v = (double)x[i];
        double r = 0.0;
        if (fabs(v) > rcond) r = (op == GTN_EW_INV) ? 1.0 / v : (op == GTN_EW_EXP ? exp(v) : pow(v, p));
        x[i] = (T)r;
    }
}

struct OddArgs {
    int32_t ndim;
    uint32_t dims[GTN_PERM_MAX_AX];
    int32_t ferm_mask, pp_mask;
    uint64_t parity;  // MASK: the parity of an entry is that of these bits of its flat index
};
template <typename I>
__device__ __forceinline__ uint32_t odd_entry(const OddArgs &a, I r) {
    uint32_t par = 0;
    for (int ax = a.ndim - 1; ax >= 0; --ax) {
        const I d = (I)a.dims[ax], k = r % d;
        r /= d;
        if ((a.ferm_mask >> ax) & 1) par ^= ((a.pp_mask >> ax) & 1) ? (uint32_t)(k & 1) : (popc64(k) & 1u);
    }
    return par;
}
// Sum of squares of the odd entries, V of them per 16-byte load.  A read of the whole tensor, and bound by
// that where every axis up to the last fermionic one is a power of two (MASK: fermionic legs always are, so
// only a bosonic leg behind one is not): a 64 x 64 x 64 x 64 tensor takes 27 us, with an index
// division an axis and 8-byte loads 54 for two axes.
template <typename T, int V, bool MASK>
__global__ void k_odd_partial(OddArgs a, const T *__restrict__ x, int64_t n, double *part) {
    __shared__ double sh[16];
    struct alignas(V * sizeof(T)) Vec {
        T v[V];
    };
    double acc = 0;
    const bool narrow = n < ((int64_t)1 << 32);
#pragma unroll 4
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n / V; i += (int64_t)gridDim.x * blockDim.x) {
        const Vec w = ((const Vec *)x)[i];
#pragma unroll
        for (int u = 0; u < V; ++u) {
            const uint64_t e = (uint64_t)i * V + u;
            const uint32_t par = MASK ? popc64(e & a.parity) & 1u
                                      : (narrow ? odd_entry<uint32_t>(a, (uint32_t)e) : odd_entry<uint64_t>(a, e));
            acc += par ? sq(w.v[u]) : 0.0;
        }
    }
    double t = block_sum(acc, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

template <typename T>
__global__ void k_axpby(const T *x, const T *y, T *out, int64_t n, double a, double b) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = (T)(a * (double)x[i] + (y ? b * (double)y[i] : 0.0));
}
__global__ void k_axpby_c(const double2 *x, const double2 *y, double2 *out, int64_t n, double ar, double ai, double br,
                          double bi) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        double2 u = x[i], r;
        r.x = ar * u.x - ai * u.y;
        r.y = ar * u.y + ai * u.x;
        if (y) {
            double2 v = y[i];
            r.x += br * v.x - bi * v.y;
            r.y += br * v.y + bi * v.x;
        }
        out[i] = r;
    }
}

// Partial sums of the two-pass reductions: 1024 doubles per (device, stream), so that reductions
// queued on different streams never share a buffer.  Kept for the life of the process.
static std::mutex g_part_mu;
static std::map<std::pair<int, hipStream_t>, double *> g_partials;
static int partial_buffer(hipStream_t s, double **p) {
    int dev;
    GTN_CHECK_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> l(g_part_mu);
    double *&b = g_partials[std::make_pair(dev, s)];
    if (!b) GTN_CHECK_HIP(hipMalloc(&b, 1024 * sizeof(double)));
    *p = b;
    return GTN_OK;
}

}  // namespace gtn

using namespace gtn;

extern "C" {

int gtn_version(void) { return 100; }

int gtn_set_dry_run(int n, const uint64_t *bases, const int64_t *bytes) {
    g_regions.clear();
    for (int i = 0; i < n; ++i) g_regions.push_back({bases[i], (uint64_t)bytes[i]});
    g_dry = n > 0;
    return GTN_OK;
}
const char *gtn_last_error(void) { return gtn::g_err; }

int gtn_device_info(char *name, int name_len, int *n_cu) {
    int dev;
    GTN_CHECK_HIP(hipGetDevice(&dev));
    hipDeviceProp_t p;
    GTN_CHECK_HIP(hipGetDeviceProperties(&p, dev));
    if (name && name_len > 0) snprintf(name, name_len, "%s", p.gcnArchName);
    if (n_cu) *n_cu = p.multiProcessorCount;
    if (strncmp(p.gcnArchName, "gfx950", 6) != 0) {
        set_error("gtn_device_info: device is %s, this library is built for gfx950", p.gcnArchName);
        return GTN_ENOTSUP;
    }
    return GTN_OK;
}

int gtn_index_tables(int64_t n, int32_t *popc, int8_t *sigma, int32_t *enc, void *stream) {
    GTN_REQUIRE(n >= 0, "gtn_index_tables: n < 0");
    if (n == 0) return GTN_OK;
    GTN_RANGE(popc, popc ? n * 4 : 0, "index_tables popc");
    GTN_RANGE(sigma, sigma ? n : 0, "index_tables sigma");
    GTN_RANGE(enc, enc ? n * 4 : 0, "index_tables enc");
    if (dry_run()) return GTN_OK;
    hipLaunchKernelGGL(k_index_tables, dim3(grid_for(n, 256)), dim3(256), 0, as_stream(stream), n, popc, sigma, enc);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

// The descriptor with every output axis that runs over several components of its virtual axis (a fused
// index, or the half of one) cut at their boundaries, so that each leg is an axis of its own for the
// tiles: an index c of stride m in V is (c / q, c % q) with strides m q and m.  Same elements, same order.
static gtn_perm_desc split_axes(const gtn_perm_desc *d) {
    gtn_perm_desc x = *d;
    int n = 0;
    int first[AX];
    for (int v = 0, j = 0; v < d->n_virt; ++v) {
        first[v] = j;
        j += d->virt_ncomp[v];
    }
    int64_t dim[AX], mul[AX][2];
    int32_t vid[AX][2];
    for (int ax = 0; ax < d->n_out; ++ax) {
        int64_t cuts[NC];
        int nc = 0;
        const int v = d->out_virt[ax][0];
        const int64_t m = d->out_vmul[ax][0];
        if (v >= 0 && d->out_virt[ax][1] < 0 && m > 0) {
            int64_t pc = 1;
            for (int j = d->virt_ncomp[v] - 1; j > 0; --j) {
                pc *= d->comp_dim[first[v] + j];
                if (pc > m && pc % m == 0 && d->out_dim[ax] % (pc / m) == 0 && pc / m < d->out_dim[ax]) cuts[nc++] = pc / m;
            }
        }
        int64_t rest = d->out_dim[ax];
        for (int c = nc - 1; c >= -1; --c) {
            const int64_t below = c >= 0 ? cuts[c] : 1;
            if (n == AX) return *d;
            dim[n] = rest / below;
            vid[n][0] = v;
            vid[n][1] = d->out_virt[ax][1];
            mul[n][0] = m * below;
            mul[n][1] = d->out_vmul[ax][1];
            rest = below;
            ++n;
        }
    }
    // every original axis may still follow: all fit
    x.n_out = n;
    for (int i = 0; i < n; ++i) {
        x.out_dim[i] = dim[i];
        for (int t = 0; t < 2; ++t) x.out_virt[i][t] = vid[i][t], x.out_vmul[i][t] = mul[i][t];
    }
    return x;
}

// Source offset of an output element on the host (the index map of perm_map without its signs).
static int64_t host_offset(const gtn_perm_desc *d, const int64_t *o) {
    auto enc = [](uint64_t i) { return i ^ (uint64_t)(__builtin_popcountll(i >> 1) & 1); };
    uint64_t V[AX] = {0}, F[AX] = {0};
    for (int ax = 0; ax < d->n_out; ++ax)
        for (int t = 0; t < 2; ++t)
            if (d->out_virt[ax][t] >= 0) V[d->out_virt[ax][t]] += (uint64_t)(o[ax] * d->out_vmul[ax][t]);
    int j = d->n_comp;
    for (int v = d->n_virt - 1; v >= 0; --v) {
        uint64_t c = d->virt_enc[v] ? enc(V[v]) : V[v];
        for (int t = 0; t < d->virt_ncomp[v]; ++t) {
            --j;
            const uint64_t k = c % (uint64_t)d->comp_dim[j];
            c /= (uint64_t)d->comp_dim[j];
            for (int u = 0; u < 2; ++u)
                if (d->comp_in[j][u] >= 0) F[d->comp_in[j][u]] += k * (uint64_t)d->comp_mult[j][u];
        }
    }
    int64_t off = 0;
    for (int b = 0; b < d->n_in; ++b) {
        const uint64_t e = d->in_enc[b] ? enc(F[b]) : F[b];
        off += d->in_split[b] ? (int64_t)(e & 1) * d->in_stride_lo[b] + (int64_t)(e >> 1) * d->in_stride[b]
                              : (int64_t)e * d->in_stride[b];
    }
    return off;
}

// 128-byte source lines that 64 consecutive steps touch: along output axis `ax` alone, or (ax < 0) of the
// output elements 0 .. 63; scaled to 64 steps.
static int lines_of(const gtn_perm_desc *d, int ax, int es) {
    int64_t o[AX] = {0}, seen[64];
    int n = 0, steps = 0;
    for (; steps < 64; ++steps) {
        if (ax >= 0) {
            if (steps >= d->out_dim[ax]) break;
            o[ax] = steps;
        } else {
            int64_t rest = steps;
            for (int x = d->n_out - 1; x >= 0; --x) {
                o[x] = rest % d->out_dim[x];
                rest /= d->out_dim[x];
            }
            if (rest) break;
        }
        const int64_t line = host_offset(d, o) * es / 128;
        int k = 0;
        while (k < n && seen[k] != line) ++k;
        if (k == n) seen[n++] = line;
    }
    return steps ? n * 64 / steps : 64;
}

// Tiles pay where 64 consecutive output elements touch more than 16 source lines (a lane group's read
// then takes a cycle per line, and lines are fetched again and again) and along some other axis of at
// least 16 indices 64 steps touch at most a third of that.
static bool plan_tiles(const gtn_perm_desc *d, TileArgs &t) {
    const int n = d->n_out, es = d->dtype == GTN_F32 ? 4 : 8;
    if (n < 2) return false;
    const int t0 = n - 1;
    if (d->out_dim[t0] < 16) return false;
    const int flat = lines_of(d, -1, es);
    if (flat <= 16) return false;
    int t1 = -1, best = flat / 3 + 1;
    for (int ax = 0; ax < t0; ++ax) {
        if (d->out_dim[ax] < 16) continue;
        const int la = lines_of(d, ax, es);
        if (la < best) {
            best = la;
            t1 = ax;
        }
    }
    if (t1 < 0) return false;
    memset(&t, 0, sizeof(t));
    t.t0 = t0;
    t.t1 = t1;
    t.sh0 = d->out_dim[t0] >= 64 ? 6 : (d->out_dim[t0] >= 32 ? 5 : 4);
    t.sh1 = d->out_dim[t1] >= 64 ? 6 : (d->out_dim[t1] >= 32 ? 5 : 4);
    int64_t acc = 1;
    for (int ax = n - 1; ax >= 0; --ax) {
        t.ostr[ax] = acc;
        acc *= d->out_dim[ax];
    }
    t.rest_total = 1;
    for (int ax = 0; ax < n; ++ax)
        if (ax != t0 && ax != t1) {
            t.rest_ax[t.n_rest++] = ax;
            t.rest_total *= d->out_dim[ax];
        }
    t.tiles0 = (int32_t)((d->out_dim[t0] + (1 << t.sh0) - 1) >> t.sh0);
    t.tiles1 = (int32_t)((d->out_dim[t1] + (1 << t.sh1) - 1) >> t.sh1);
    return (int64_t)t.tiles0 * t.tiles1 * t.rest_total < (1 << 30);
}

// Group the virtual axes for the table-driven map (k_perm_tables).  Returns false when the gather
// is so small that one wavefront walks it, or a group's table would be large: the table is built once per
// gather shape (about 20 us), and every gather without one walks the descriptor with its index vectors in
// scratch memory, 12 to 20 us for the smallest (MI355X; 5 us with tables).
// `fast`: the output axis whose index runs fastest in the tables (-1: the last one that feeds the group).
static bool plan_groups(const gtn_perm_desc *d, int64_t total, int fast, TabBuild &tb, TabArgs &ta) {
    if (total < 64 || d->n_virt == 0) return false;
    const int nv = d->n_virt;
    // the virtual axis that feeds each input axis (-1: none, -2: several), and whether the map is linear
    // over GF(2)
    bool lin = true;
    {
        int feeder[AX];
        uint64_t fbits[AX] = {0}, used = 0;
        for (int b = 0; b < d->n_in; ++b) feeder[b] = -1;
        auto pow2 = [](int64_t x) { return x > 0 && (x & (x - 1)) == 0; };
        int jj = 0;
        for (int v = 0; v < nv; ++v)
            for (int t = 0; t < d->virt_ncomp[v]; ++t, ++jj) {
                lin = lin && pow2(d->comp_dim[jj]);
                for (int u = 0; u < 2; ++u) {
                    const int b = d->comp_in[jj][u];
                    if (b < 0) continue;
                    feeder[b] = feeder[b] == -1 || feeder[b] == v ? v : -2;
                    if (d->comp_dim[jj] == 1) continue;
                    lin = lin && pow2(d->comp_mult[jj][u]);
                    const uint64_t bits = (uint64_t)(d->comp_dim[jj] - 1) * (uint64_t)d->comp_mult[jj][u];
                    lin = lin && !(fbits[b] & bits);
                    fbits[b] |= bits;
                }
            }
        auto take = [&](int64_t n, int64_t stride) {  // offset bits of an index of n values
            if (n <= 1 || stride == 0) return;
            const uint64_t bits = (uint64_t)(n - 1) * (uint64_t)stride;
            lin = lin && pow2(n) && pow2(stride) && !(used & bits);
            used |= bits;
        };
        for (int b = 0; b < d->n_in && lin; ++b) {
            lin = pow2(d->in_dim[b]) && !(d->in_sigma[b] && feeder[b] == -2);
            if (d->in_split[b]) {
                take(2 < d->in_dim[b] ? 2 : d->in_dim[b], d->in_stride_lo[b]);
                take(d->in_dim[b] >> 1, d->in_stride[b]);
            } else {
                take(d->in_dim[b], d->in_stride[b]);
            }
        }
    }
    // union virtual axes whose components feed a common input axis (a linear map needs no union)
    int parent[AX];
    for (int v = 0; v < nv; ++v) parent[v] = v;
    auto root = [&](int v) {
        while (parent[v] != v) v = parent[v];
        return v;
    };
    int owner[AX];
    uint32_t feeds[AX] = {0};  // input axes fed by each virtual axis
    for (int b = 0; b < d->n_in; ++b) owner[b] = -1;
    int j = 0;
    for (int v = 0; v < nv; ++v)
        for (int t = 0; t < d->virt_ncomp[v]; ++t, ++j)
            for (int u = 0; u < 2; ++u) {
                const int b = d->comp_in[j][u];
                if (b < 0) continue;
                feeds[v] |= 1u << b;
                if (owner[b] < 0)
                    owner[b] = v;
                else if (!lin)
                    parent[root(v)] = root(owner[b]);
            }
    // groups in order of their smallest virtual axis; a group's table has an entry for every value of the
    // output axes that feed one of its virtual axes
    int gid[AX], ng = 0;
    uint32_t members[AX];
    auto fed = [&](uint32_t mem, int ax) {
        for (int t = 0; t < 2; ++t)
            if (d->out_virt[ax][t] >= 0 && (mem >> d->out_virt[ax][t] & 1u)) return true;
        return false;
    };
    auto size_of = [&](uint32_t mem) -> int64_t {
        int64_t n = 1;
        for (int ax = 0; ax < d->n_out; ++ax)
            if (fed(mem, ax) && (n *= d->out_dim[ax]) > (1 << 22)) break;
        return n;
    };
    for (int v = 0; v < nv; ++v) gid[v] = -1;
    for (int v = 0; v < nv; ++v) {
        const int r = root(v);
        if (gid[r] < 0) {
            gid[r] = ng;
            members[ng++] = 0;
        }
        members[gid[r]] |= 1u << v;
        if (size_of(members[gid[r]]) > (1 << 22)) return false;
    }
    // merge the two smallest groups while there are too many
    while (ng > kTabGroups) {
        int a0 = 0, a1 = 1;
        if (size_of(members[a1]) < size_of(members[a0])) std::swap(a0, a1);
        for (int g = 2; g < ng; ++g) {
            if (size_of(members[g]) < size_of(members[a0])) {
                a1 = a0;
                a0 = g;
            } else if (size_of(members[g]) < size_of(members[a1])) {
                a1 = g;
            }
        }
        if (a1 < a0) std::swap(a0, a1);
        members[a0] |= members[a1];
        if (size_of(members[a0]) > (1 << 22)) return false;
        for (int g = a1; g + 1 < ng; ++g) members[g] = members[g + 1];
        --ng;
    }
    int64_t entries = 0;
    for (int g = 0; g < ng; ++g) entries += size_of(members[g]);
    if (entries > (total < (1 << 16) ? total : total / 4)) return false;
    memset(&tb, 0, sizeof(tb));
    memset(&ta, 0, sizeof(ta));
    tb.ng = ta.ng = ng;
    ta.lin = lin;
    for (int g = 0; g < ng; ++g) {
        tb.start[g + 1] = tb.start[g] + size_of(members[g]);
        tb.vmask[g] = members[g];
        for (int v = 0; v < nv; ++v)
            if (members[g] >> v & 1u) tb.inmask[g] |= feeds[v];
        int64_t rad = 1;
        for (int i = d->n_out; i >= 0; --i) {  // axis `fast` first, then the output's from the last
            const int ax = i == d->n_out ? fast : i;
            if (ax < 0 || (i < d->n_out && ax == fast) || !fed(members[g], ax)) continue;
            tb.ax[g][tb.nx[g]] = (int8_t)ax;
            tb.rad[g][tb.nx[g]++] = (uint32_t)rad;
            ta.gmul[ax][g] = (uint32_t)rad;
            rad *= d->out_dim[ax];
        }
    }
    return true;
}

// Device tables of the table-driven map, built once per gather shape and device and kept until
// the cache outgrows kTabCacheBytes (then every table is released after a device synchronisation).
struct TabCacheEntry {
    TabEntry *dev;
    int64_t entries;
};
// shared from a gather's look-up to its launch, exclusive while tables are built and dropped: a table that a
// launch has been given is not released before that launch is on its stream
static std::shared_mutex g_tab_mu;
static std::mutex g_tab_turn;  // passed on the way in, and kept by who builds: launches do not keep it waiting forever
static std::map<std::string, TabCacheEntry> g_tab_cache;
static int64_t g_tab_bytes = 0;
constexpr int64_t kTabCacheBytes = 64ll << 20;
constexpr int64_t kTabSlab = 1 << 20;
struct TabStore {
    char *next = nullptr;
    int64_t left = 0;
};
static std::map<int, TabStore> g_tab_store;      // per device: the slab being cut
static std::vector<void *> g_tab_slabs;
static std::map<int, hipStream_t> g_tab_stream;  // per device: the stream tables are built on

// one gather's tables: what they are made from, and where their addresses go
struct TabWant {
    const PermArgs *a;
    const TabBuild *build;
    TabArgs *out;
    std::string key;
};
// held until the launch
struct TabHold {
    std::unique_lock<std::mutex> turn;
    std::shared_lock<std::shared_mutex> shared;
    std::unique_lock<std::shared_mutex> exclusive;
};

static int64_t tab_bytes(const TabBuild &b) { return (b.start[b.ng] * (int64_t)sizeof(TabEntry) + 255) / 256 * 256; }

static int build_table(const TabWant &w, int dev) {
    // tables are cut from slabs, one at a time in use per device; the build stream is kept with it
    TabStore &store = g_tab_store[dev];
    const int64_t n = w.build->start[w.build->ng], bytes = tab_bytes(*w.build);
    if (store.left < bytes) {
        const int64_t slab = bytes > kTabSlab ? bytes : kTabSlab;
        void *p = nullptr;
        GTN_CHECK_HIP(hipMalloc(&p, slab));
        g_tab_slabs.push_back(p);
        store.next = (char *)p;
        store.left = slab;
    }
    hipStream_t &bs = g_tab_stream[dev];
    if (!bs) GTN_CHECK_HIP(hipStreamCreateWithFlags(&bs, hipStreamNonBlocking));
    // built on a stream of their own and finished here: the tables are shared by later gathers
    // on any stream, and the caller's stream may be capturing a graph
    TabEntry *p = (TabEntry *)store.next;
    hipLaunchKernelGGL(k_perm_tables, dim3(grid_for(n, 256, 4096)), dim3(256), 0, bs, *w.a, *w.build, p);
    GTN_CHECK_HIP(hipGetLastError());
    GTN_CHECK_HIP(hipStreamSynchronize(bs));
    store.next += bytes;
    store.left -= bytes;
    g_tab_cache.emplace(w.key, TabCacheEntry{p, n});
    g_tab_bytes += bytes;
    return GTN_OK;
}

static bool tab_find(const TabWant &w) {
    auto it = g_tab_cache.find(w.key);
    if (it == g_tab_cache.end()) return false;
    for (int g = 0; g < w.build->ng; ++g) w.out->tab[g] = it->second.dev + w.build->start[g];
    return true;
}

// The tables of `count` gathers (of one launch), built where they are not there yet; `hold` has to outlive the launch.
static int tab_tables(TabWant *want, int count, TabHold &hold) {
    int dev;
    GTN_CHECK_HIP(hipGetDevice(&dev));
    for (int i = 0; i < count; ++i) {
        PermArgs k;
        memcpy(&k, want[i].a, sizeof(k));
        memset(k.table, 0, sizeof(k.table));
        k.alpha_re = k.alpha_im = 0.0;
        want[i].key.assign((const char *)&dev, sizeof(dev));
        want[i].key.append((const char *)&k, sizeof(k));
        want[i].key.append((const char *)want[i].build, sizeof(TabBuild));
    }
    hold.turn = std::unique_lock<std::mutex>(g_tab_turn);
    hold.shared = std::shared_lock<std::shared_mutex>(g_tab_mu);
    hold.turn.unlock();
    bool there = true;
    for (int i = 0; i < count; ++i) there = tab_find(want[i]) && there;
    if (there) return GTN_OK;
    hold.shared.unlock();
    hold.turn.lock();
    hold.exclusive = std::unique_lock<std::shared_mutex>(g_tab_mu);
    int64_t more = 0;
    for (int i = 0; i < count; ++i) more += tab_find(want[i]) ? 0 : tab_bytes(*want[i].build);
    // over budget: drop the cache, unless a graph may hold some of its tables
    if (more && g_tab_bytes + more > kTabCacheBytes && !g_tab_cache.empty() && !graphs_alive() && !capture_open()) {
        GTN_CHECK_HIP(hipDeviceSynchronize());
        g_tab_store.clear();
        g_tab_cache.clear();
        g_tab_bytes = 0;
        std::vector<void *> slabs;
        slabs.swap(g_tab_slabs);
        for (void *slab : slabs) GTN_CHECK_HIP(hipFree(slab));
    }
    for (int i = 0; i < count; ++i) {
        if (tab_find(want[i])) continue;
        int rc = build_table(want[i], dev);
        if (rc) return rc;
        (void)tab_find(want[i]);
    }
    return GTN_OK;
}

// GTN_PERM_TILED=0 in the environment turns the LDS-tiled gather off (tuning and tests).
static bool tiles_enabled() {
    static int on = -1;
    if (on < 0) {
        const char *e = getenv("GTN_PERM_TILED");
        on = (e && atoi(e) == 0) ? 0 : 1;
    }
    return on == 1;
}

// Row walk (k_permute_rows) where some trailing axes make rows of whole chunks; a last axis that is no power
// of two needs three axes and more for that, and a division a column (32^4 x 9 doubles: 64 us by
// k_permute's walk, 35 by rows).  1024-column chunks for
// gathers that still fill the device with them (four loads in flight per lane), 256 otherwise.  Each
// workgroup takes up to 8 rows once there are more than 16 workgroups per compute unit without that, and more
// where the grid would exceed kMaxGrid.
static bool plan_rows(const PermArgs &a, const TabArgs &tb, RowArgs &w, int &U) {
    U = a.total >= (1 << 20) ? 4 : 1;
    for (;; U = 1) {
        const int64_t chunk = U * 256;
        int64_t width = 1;
        for (int ns = 1; ns <= a.n_out; ++ns) {
            const int ax = a.n_out - ns;
            width *= a.out_dim[ax];
            if (width >= ((int64_t)1 << 32)) break;
            if (width % chunk) continue;
            w.width = width;
            w.rows = a.total / width;
            w.ns = ns;
            w.chunks = (int32_t)(width / chunk);
            const int64_t per = w.rows * w.chunks / 4096, least = (w.rows * w.chunks + kMaxGrid - 1) / kMaxGrid;
            w.rows_per = (int32_t)std::max<int64_t>(per < 1 ? 1 : (per > 8 ? 8 : per), least);
            if ((w.rows + w.rows_per - 1) / w.rows_per * w.chunks >= 2 * kMaxGrid) return false;
            w.vary = 0;
            for (int k = 0; k < ns; ++k)
                for (int g = 0; g < tb.ng; ++g)
                    if (tb.gmul[a.n_out - 1 - k][g]) w.vary |= 1u << g;
            return true;
        }
        if (U == 1) return false;
    }
}

// What gtn_permute does with a descriptor, planned once per gather shape (the sign table, alpha and the
// size of the source aside) and device.
struct PermPlan {
    bool tab, tile, rows;
    PermArgs a;  // of the descriptor the kernels walk; sign table and alpha filled in per call
    TabBuild build;
    TabArgs tb;
    TileArgs t;
    RowArgs w;
    int U;
};
static std::mutex g_plan_mu;
static std::map<std::string, PermPlan> g_plans;
constexpr size_t kMaxPlans = 4096;

static int plan_permute(const gtn_perm_desc *d, PermArgs &a, PermPlan &p) {
    memset(&p, 0, sizeof(p));
    const bool fp = d->dtype == GTN_F64 || d->dtype == GTN_F32;
    p.a = a;
    if (!fp) return GTN_OK;
    const gtn_perm_desc x = split_axes(d);
    PermArgs ax;
    int rc = build_perm_args(&x, ax);
    if (rc) return rc;
    p.tile = tiles_enabled() && plan_tiles(&x, p.t);
    p.tab = getenv("GTN_PERM_NO_TABLES") == nullptr && plan_groups(&x, ax.total, p.tile ? p.t.t1 : -1, p.build, p.tb);
    p.a = ax;
    p.rows = p.tab && !p.tile && plan_rows(p.a, p.tb, p.w, p.U);
    return GTN_OK;
}

int gtn_permute(const gtn_perm_desc *d, const void *src, void *dst, void *stream) {
    GTN_REQUIRE(d && src && dst, "gtn_permute: null argument");
    PermArgs a;
    int rc = build_perm_args(d, a);
    if (rc) return rc;
    if (a.total == 0) return GTN_OK;
    if (dry_run()) {
        int es = d->dtype == GTN_C128 ? 16 : (d->dtype == GTN_F32 ? 4 : 8);
        GTN_RANGE(src, d->src_elems * es, "permute src");
        GTN_RANGE(dst, a.total * es, "permute dst");
        return GTN_OK;
    }
    hipStream_t s = as_stream(stream);
    PermPlan p;
    {
        PermArgs k;
        memcpy(&k, &a, sizeof(k));
        memset(k.table, 0, sizeof(k.table));
        k.alpha_re = k.alpha_im = 0.0;
        const int32_t kind[2] = {d->dtype, getenv("GTN_PERM_NO_TABLES") != nullptr};
        std::string key((const char *)kind, sizeof(kind));
        key.append((const char *)&k, sizeof(k));
        std::lock_guard<std::mutex> l(g_plan_mu);
        auto it = g_plans.find(key);
        if (it == g_plans.end()) {
            rc = plan_permute(d, a, p);
            if (rc) return rc;
            if (g_plans.size() >= kMaxPlans) g_plans.clear();
            it = g_plans.emplace(std::move(key), p).first;
        }
        p = it->second;
    }
    memcpy(p.a.table, a.table, sizeof(a.table));
    p.a.alpha_re = a.alpha_re;
    p.a.alpha_im = a.alpha_im;
    p.tb.signs = (uint64_t)d->table[0] | (uint64_t)d->table[1] << 32;
    p.tb.short_signs = d->n_bits <= 5;
    TabHold hold;
    if (p.tab) {
        TabWant want{&p.a, &p.build, &p.tb, {}};
        rc = tab_tables(&want, 1, hold);
        if (rc) return rc;
    }
    if (p.tile) {
        TileArgs &t = p.t;
        const int64_t nblk = (int64_t)t.tiles0 * t.tiles1 * t.rest_total;
        const size_t lds = sizeof(double) * ((size_t)1 << t.sh1) * ((1 << t.sh0) + 1);
        // kMaxGrid tiles a launch, an eighth of them of each XCD's share
        for (int64_t done = 0; done < (nblk + 7) / 8; done += kMaxGrid / 8) {
            t.slot0 = (uint32_t)done;
            const dim3 gt((unsigned)(8 * std::min((nblk + 7) / 8 - done, kMaxGrid / 8))), bt(256);
#define GTN_TILES(T, B) \
    hipLaunchKernelGGL((k_permute_tiled<T, B>), gt, bt, lds, s, p.a, p.tb, t, (const T *)src, (T *)dst)
            if (d->dtype == GTN_F64) {
                if (p.tab) GTN_TILES(double, true);
                else GTN_TILES(double, false);
            } else {
                if (p.tab) GTN_TILES(float, true);
                else GTN_TILES(float, false);
            }
#undef GTN_TILES
            GTN_CHECK_LAUNCH();
        }
        return GTN_OK;
    }
    if (p.rows) {
        const RowArgs &w = p.w;
        const dim3 gr((unsigned)((w.rows + w.rows_per - 1) / w.rows_per * w.chunks)), br(256);
#define GTN_ROWS(T, N) hipLaunchKernelGGL((k_permute_rows<T, N>), gr, br, 0, s, p.a, p.tb, w, (const T *)src, (T *)dst)
        if (d->dtype == GTN_F64) {
            if (p.U == 4) GTN_ROWS(double, 4);
            else GTN_ROWS(double, 1);
        } else {
            if (p.U == 4) GTN_ROWS(float, 4);
            else GTN_ROWS(float, 1);
        }
#undef GTN_ROWS
        GTN_CHECK_LAUNCH();
        return GTN_OK;
    }
    dim3 g(grid_for((a.total + kPermUnroll - 1) / kPermUnroll, 256, 1 << 20)), b(256);
#define GTN_WALK(T, B) hipLaunchKernelGGL((k_permute<T, B>), g, b, 0, s, p.a, p.tb, (const T *)src, (T *)dst)
    switch (d->dtype) {
        case GTN_F64:
            if (p.tab) GTN_WALK(double, true);
            else GTN_WALK(double, false);
            break;
        case GTN_F32:
            if (p.tab) GTN_WALK(float, true);
            else GTN_WALK(float, false);
            break;
        case GTN_C128: hipLaunchKernelGGL(k_permute_c128, g, b, 0, s, a, (const double2 *)src, (double2 *)dst); break;
        default: set_error("gtn_permute: unsupported dtype %d", d->dtype); return GTN_ENOTSUP;
    }
#undef GTN_WALK
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_permute2(const gtn_perm_desc *outer, const gtn_perm_desc *inner, const void *src, void *dst, void *stream) {
    GTN_REQUIRE(outer && inner && src && dst, "gtn_permute2: null argument");
    GTN_REQUIRE(outer->dtype == inner->dtype && (outer->dtype == GTN_F64 || outer->dtype == GTN_F32),
                "gtn_permute2: both gathers must be F64 or both F32");
    PermArgs ao, an;
    int rc = build_perm_args(outer, ao);
    if (rc) return rc;
    rc = build_perm_args(inner, an);
    if (rc) return rc;
    GTN_REQUIRE(outer->src_elems == an.total, "gtn_permute2: the outer gather reads %lld elements, the inner one makes %lld",
                (long long)outer->src_elems, (long long)an.total);
    if (ao.total == 0) return GTN_OK;
    if (dry_run()) {
        const int es = outer->dtype == GTN_F32 ? 4 : 8;
        GTN_RANGE(src, inner->src_elems * es, "permute2 src");
        GTN_RANGE(dst, ao.total * es, "permute2 dst");
        return GTN_OK;
    }
    hipStream_t s = as_stream(stream);
    TabArgs to, tn;
    memset(&to, 0, sizeof(to));
    memset(&tn, 0, sizeof(tn));
    TabBuild bo, bn;
    const bool tabs = getenv("GTN_PERM_NO_TABLES") == nullptr;
    const bool tabo = tabs && plan_groups(outer, ao.total, -1, bo, to);
    const bool tabn = tabs && plan_groups(inner, an.total, -1, bn, tn);
    to.signs = (uint64_t)outer->table[0] | (uint64_t)outer->table[1] << 32;
    tn.signs = (uint64_t)inner->table[0] | (uint64_t)inner->table[1] << 32;
    to.short_signs = outer->n_bits <= 5;
    tn.short_signs = inner->n_bits <= 5;
    TabWant want[2];
    int wants = 0;
    if (tabo) want[wants++] = TabWant{&ao, &bo, &to, {}};
    if (tabn) want[wants++] = TabWant{&an, &bn, &tn, {}};
    TabHold hold;
    if (wants && (rc = tab_tables(want, wants, hold))) return rc;
    dim3 g(grid_for((ao.total + kPermUnroll - 1) / kPermUnroll, 256, 1 << 20)), b(256);
#define GTN_P2(T, A, B) hipLaunchKernelGGL((k_permute2<T, A, B>), g, b, 0, s, ao, to, an, tn, (const T *)src, (T *)dst)
    if (outer->dtype == GTN_F64) {
        if (tabo && tabn) GTN_P2(double, true, true);
        else if (tabo) GTN_P2(double, true, false);
        else if (tabn) GTN_P2(double, false, true);
        else GTN_P2(double, false, false);
    } else {
        if (tabo && tabn) GTN_P2(float, true, true);
        else if (tabo) GTN_P2(float, true, false);
        else if (tabn) GTN_P2(float, false, true);
        else GTN_P2(float, false, false);
    }
#undef GTN_P2
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_sign_tensor(int ndim, const int64_t *dims, const uint32_t *table, int8_t *out, void *stream) {
    GTN_REQUIRE(ndim >= 0 && ndim <= GTN_PERM_MAX_BITS, "gtn_sign_tensor: ndim out of range");
    SignArgs a;
    memset(&a, 0, sizeof(a));
    a.ndim = ndim;
    int64_t total = 1;
    for (int i = 0; i < ndim; ++i) {
        GTN_REQUIRE(dims[i] >= 1 && dims[i] < (1ll << 31), "gtn_sign_tensor: bad dim");
        a.dims[i] = (uint32_t)dims[i];
        total *= dims[i];
    }
    a.total = total;
    memcpy(a.table, table, ((1u << ndim) + 31) / 32 * sizeof(uint32_t));
    hipLaunchKernelGGL(k_sign_tensor, dim3(grid_for(total, 256, 1 << 20)), dim3(256), 0, as_stream(stream), a, out);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_sumsq(const void *x, int64_t n, int dtype, double *out, void *stream) {
    hipStream_t s = as_stream(stream);
    double *part;
    int rc = partial_buffer(s, &part);
    if (rc) return rc;
    int g = grid_for(n, 256, 1024);
    switch (dtype) {
        case GTN_F64: hipLaunchKernelGGL(k_sumsq_partial<double>, dim3(g), dim3(256), 0, s, (const double *)x, n, part); break;
        case GTN_F32: hipLaunchKernelGGL(k_sumsq_partial<float>, dim3(g), dim3(256), 0, s, (const float *)x, n, part); break;
        case GTN_C128: hipLaunchKernelGGL(k_sumsq_partial<double2>, dim3(g), dim3(256), 0, s, (const double2 *)x, n, part); break;
        default: set_error("gtn_sumsq: unsupported dtype"); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_sum_final, dim3(1), dim3(1024), 0, s, (const double *)part, g, out);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_scale_by_norm(void *x, int64_t n, int dtype, const double *nrm2, void *stream) {
    hipStream_t s = as_stream(stream);
    dim3 g(grid_for(n, 256, 1 << 16)), b(256);
    switch (dtype) {
        case GTN_F64: hipLaunchKernelGGL(k_scale_by_norm<double>, g, b, 0, s, (double *)x, n, nrm2); break;
        case GTN_F32: hipLaunchKernelGGL(k_scale_by_norm<float>, g, b, 0, s, (float *)x, n, nrm2); break;
        case GTN_C128: hipLaunchKernelGGL(k_scale_by_norm_c, g, b, 0, s, (double2 *)x, n, nrm2); break;
        default: set_error("gtn_scale_by_norm: unsupported dtype"); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_reduce_last(const void *src, void *dst, int64_t rows, int64_t inner, int dtype, void *stream) {
    hipStream_t s = as_stream(stream);
    dim3 g(grid_for(rows, 256, 1 << 16)), b(256);
    switch (dtype) {
        case GTN_F64: hipLaunchKernelGGL(k_reduce_last<double>, g, b, 0, s, (const double *)src, (double *)dst, rows, inner); break;
        case GTN_F32: hipLaunchKernelGGL(k_reduce_last<float>, g, b, 0, s, (const float *)src, (float *)dst, rows, inner); break;
        case GTN_C128: hipLaunchKernelGGL(k_reduce_last_c, g, b, 0, s, (const double2 *)src, (double2 *)dst, rows, inner); break;
        default: set_error("gtn_reduce_last: unsupported dtype"); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_lognorm_update(double *ln, const double *nrm2, void *stream) {
    hipLaunchKernelGGL(k_lognorm, dim3(1), dim3(64), 0, as_stream(stream), ln, nrm2);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_power_diag(void *x, int64_t n, int64_t stride, int dtype, double p, double rcond, void *stream) {
    hipStream_t s = as_stream(stream);
    dim3 g(grid_for(n, 256)), b(256);
    switch (dtype) {
        case GTN_F64: hipLaunchKernelGGL(k_power_diag<double>, g, b, 0, s, (double *)x, n, stride, p, rcond); break;
        case GTN_F32: hipLaunchKernelGGL(k_power_diag<float>, g, b, 0, s, (float *)x, n, stride, p, rcond); break;
        default: set_error("gtn_power_diag: unsupported dtype"); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_elementwise(void *x, int64_t n, int dtype, int op, double p, double rcond, void *stream) {
    GTN_REQUIRE(n >= 0 && (n == 0 || x), "gtn_elementwise: bad buffer");
    GTN_REQUIRE(op == GTN_EW_POWER || op == GTN_EW_INV || op == GTN_EW_EXP, "gtn_elementwise: unknown op %d", op);
    if (n == 0) return GTN_OK;
    hipStream_t s = as_stream(stream);
    dim3 g(grid_for(n, 256)), b(256);
    switch (dtype) {
        case GTN_F64: hipLaunchKernelGGL(k_elementwise<double>, g, b, 0, s, (double *)x, n, op, p, rcond); break;
        case GTN_F32: hipLaunchKernelGGL(k_elementwise<float>, g, b, 0, s, (float *)x, n, op, p, rcond); break;
        default: set_error("gtn_elementwise: unsupported dtype"); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_axpby(const void *x, const void *y, void *out, int64_t n, int dtype, double ar, double ai, double br, double bi,
              void *stream) {
    if (n == 0) return GTN_OK;
    hipStream_t s = as_stream(stream);
    dim3 g(grid_for(n, 256, 1 << 16)), b(256);
    switch (dtype) {
        case GTN_F64: hipLaunchKernelGGL(k_axpby<double>, g, b, 0, s, (const double *)x, (const double *)y, (double *)out, n, ar, br); break;
        case GTN_F32: hipLaunchKernelGGL(k_axpby<float>, g, b, 0, s, (const float *)x, (const float *)y, (float *)out, n, ar, br); break;
        case GTN_C128:
            hipLaunchKernelGGL(k_axpby_c, g, b, 0, s, (const double2 *)x, (const double2 *)y, (double2 *)out, n, ar, ai, br, bi);
            break;
        default: set_error("gtn_axpby: unsupported dtype"); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_normalize_batch(void *x, void *dst, int64_t nbatch, int64_t n, int dtype, double *nrm2, double *lognorm,
                        double *hist, int hist_len, double *step, void *stream) {
    GTN_REQUIRE(nbatch >= 1 && nbatch <= 1024 && n >= 1, "gtn_normalize_batch: need 1 <= nbatch <= 1024 and n >= 1");
    GTN_REQUIRE(x && nrm2, "gtn_normalize_batch: null buffer");
    GTN_REQUIRE(dtype == GTN_F64 || dtype == GTN_F32, "gtn_normalize_batch: dtype must be F64 or F32");
    hipStream_t s = as_stream(stream);
    double *part;
    int rc = partial_buffer(s, &part);
    if (rc) return rc;
    const int G = (int)(1024 / nbatch) < grid_for(n, 256, 1024) ? (int)(1024 / nbatch) : grid_for(n, 256, 1024);
    const dim3 g2((unsigned)G, (unsigned)nbatch), b(256);
    if (dtype == GTN_F64)
        hipLaunchKernelGGL(k_sumsq_batch_partial<double>, g2, b, 0, s, (const double *)x, n, part);
    else
        hipLaunchKernelGGL(k_sumsq_batch_partial<float>, g2, b, 0, s, (const float *)x, n, part);
    GTN_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_norm_batch_final, dim3((unsigned)nbatch), dim3(256), 0, s, (const double *)part, G, nrm2,
                       lognorm, hist, hist_len, (const double *)step);
    GTN_CHECK_LAUNCH();
    const dim3 g3((unsigned)grid_for(n, 256, (int)(65536 / nbatch) > 0 ? (int)(65536 / nbatch) : 1), (unsigned)nbatch);
    if (!dst) dst = x;
    if (dtype == GTN_F64)
        hipLaunchKernelGGL(k_scale_batch<double>, g3, b, 0, s, (const double *)x, (double *)dst, n, (const double *)nrm2);
    else
        hipLaunchKernelGGL(k_scale_batch<float>, g3, b, 0, s, (const float *)x, (float *)dst, n, (const double *)nrm2);
    GTN_CHECK_LAUNCH();
    if (step) {
        hipLaunchKernelGGL(k_step_increment, dim3(1), dim3(64), 0, s, step);
        GTN_CHECK_LAUNCH();
    }
    return GTN_OK;
}

int gtn_diag_interleave(void *dst, int64_t nbatch, int64_t d, const void *src, int dtype, void *stream) {
    GTN_REQUIRE(nbatch >= 0 && d >= 0 && (nbatch * d == 0 || (dst && src)), "gtn_diag_interleave: bad argument");
    if (nbatch * d == 0) return GTN_OK;
    hipStream_t s = as_stream(stream);
    const int64_t total = nbatch * 4 * d * d;
    dim3 g(grid_for(total, 256, 1 << 16)), b(256);
    switch (dtype) {
        case GTN_F64: hipLaunchKernelGGL(k_diag_interleave<double>, g, b, 0, s, (double *)dst, nbatch, d, (const double *)src); break;
        case GTN_F32: hipLaunchKernelGGL(k_diag_interleave<float>, g, b, 0, s, (float *)dst, nbatch, d, (const float *)src); break;
        default: set_error("gtn_diag_interleave: dtype must be F64 or F32"); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_odd_norm(const void *x, int ndim, const int64_t *dims, const int32_t *ferm, const int32_t *pp, int dtype,
                 double *out, void *stream) {
    GTN_REQUIRE(ndim >= 0 && ndim <= GTN_PERM_MAX_AX, "gtn_odd_norm: ndim out of range");
    OddArgs a;
    memset(&a, 0, sizeof(a));
    a.ndim = ndim;
    int64_t n = 1;
    for (int i = 0; i < ndim; ++i) {
        a.dims[i] = (uint32_t)dims[i];
        n *= dims[i];
        if (ferm[i]) a.ferm_mask |= 1 << i;
        if (pp[i]) a.pp_mask |= 1 << i;
    }
    hipStream_t s = as_stream(stream);
    double *part;
    int rc = partial_buffer(s, &part);
    if (rc) return rc;
    bool mask = true;
    int64_t below = 1;  // entries of the axes behind
    for (int i = ndim - 1; i >= 0; --i) {
        const int64_t d = dims[i];
        const bool pow2 = d > 0 && (d & (d - 1)) == 0;
        if (!pow2 && (a.ferm_mask & ((2 << i) - 1))) mask = false;
        if (!mask || !pow2) break;  // (no fermionic axis is left where the last axis read was none)
        if (ferm[i] && d > 1) a.parity |= pp[i] ? (uint64_t)below : (uint64_t)below * (uint64_t)(d - 1);
        below *= d;
    }
    const int g = grid_for(n, 256, 1024);
    const dim3 grid(g), blk(256);
    auto launch = [&](auto *p, auto wide) {
        using T = std::remove_const_t<std::remove_pointer_t<decltype(p)>>;
        constexpr int V = decltype(wide)::value;
        if (mask)
            hipLaunchKernelGGL((k_odd_partial<T, V, true>), grid, blk, 0, s, a, p, n, part);
        else
            hipLaunchKernelGGL((k_odd_partial<T, V, false>), grid, blk, 0, s, a, p, n, part);
    };
    const bool al = ((uintptr_t)x & 15) == 0;
    using one = std::integral_constant<int, 1>;
    switch (dtype) {
        case GTN_F64:
            if (al && n % 2 == 0)
                launch((const double *)x, std::integral_constant<int, 2>{});
            else
                launch((const double *)x, one{});
            break;
        case GTN_F32:
            if (al && n % 4 == 0)
                launch((const float *)x, std::integral_constant<int, 4>{});
            else
                launch((const float *)x, one{});
            break;
        case GTN_C128: launch((const double2 *)x, one{}); break;
        default: set_error("gtn_odd_norm: unsupported dtype"); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_sum_final, dim3(1), dim3(1024), 0, s, (const double *)part, g, out);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

}  // extern "C"
