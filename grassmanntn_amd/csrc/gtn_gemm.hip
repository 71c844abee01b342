// Grouped, batched MFMA GEMM for the parity-block contractions (replaces oe.contract at
// __init__.py:2295 and einsum_block's per-sector np.einsum at :2781).
//
// One launch covers up to kMaxGroups independent GEMMs (the nonzero parity sectors of a
// contraction, or the parity blocks of a decomposition).  Workgroups of 256 lanes (4 wave64s in a
// 2x2 arrangement) compute a BM x BN tile; operand tiles are staged through LDS.  Precision is a
// template parameter:
//   F64    : v_mfma_f64_16x16x4f64, FP64 accumulation
//   F32    : operands rounded to FP32 on their way into LDS, v_mfma_f32_16x16x4f32
//   BF16Xn : operands split into n BF16 terms on their way into LDS (hi/lo for n=2, hi/mid/lo for
//            n=3), v_mfma_f32_16x16x32_bf16 on the 3 (n=2) or 6 (n=3) leading cross products,
//            FP32 accumulation.
// The element type in HBM stays FP64 (or FP32); the reduced precision lives only between LDS and
// the matrix cores.
#include "gtn_common.h"
#include <stdlib.h>
#include <string.h>
#include <map>
#include <mutex>
#include <vector>

namespace gtn {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int kMaxGroups = 12;

// splits > 1: the reduction dimension is cut into chunks of kchunk; the tile enumeration runs over
// batch * splits, and chunk sp of batch entry b writes its partial product to C + b * scb + sp * scs
// (a workspace summed afterwards by k_split_sum).
struct GemmGroup {
    const void *A;
    const void *B;
    void *C;
    int32_t M, N, K, batch;
    int32_t tiles_m, tiles_n;
    int32_t splits, kchunk;
    int64_t sam, sak, sbk, sbn, scm, scn, sab, sbb, scb, scs;
    double alpha, beta;
    GemmIndirect ind;  // coef null: a plain group (a launch's groups are all of one kind)
    int32_t tri;       // symmetric product: only tiles on or above the diagonal, stored on both sides of it
};

struct GemmArgs {
    int32_t n_groups;
    int32_t tile_start[kMaxGroups + 1];  // prefix sum of tiles (incl. batch) per group
    GemmGroup g[kMaxGroups];
};

// Locate this workgroup's (group, batch, tile_m, tile_n).  Tiles are enumerated per XCD in
// contiguous ranges so that workgroups sharing operand panels share an L2.
__device__ __forceinline__ bool locate(const GemmArgs &a, int &gi, int &b, int &tm, int &tn) {
    int total = a.tile_start[a.n_groups];
    int bid = blockIdx.x;
    int per = (total + 7) / 8;
    int xcd = bid % 8, slot = bid / 8;
    int t = xcd * per + slot;
    // blocks beyond `total` are launched only to round the grid to a multiple of 8
    if (t >= total) return false;
    gi = 0;
    while (gi + 1 < a.n_groups && t >= a.tile_start[gi + 1]) ++gi;
    t -= a.tile_start[gi];
    const GemmGroup &g = a.g[gi];
    int per_b = g.tri ? g.tiles_n * (g.tiles_n + 1) / 2 : g.tiles_m * g.tiles_n;
    b = t / per_b;
    t -= b * per_b;
    if (g.tri) {  // rows of tiles_n, tiles_n - 1, ... tiles
        tm = 0;
        while (t >= g.tiles_n - tm) t -= g.tiles_n - tm++;
        tn = tm + t;
        return true;
    }
    tm = t / g.tiles_n;
    tn = t - tm * g.tiles_n;
    return true;
}

template <typename T>
__device__ __forceinline__ double ld(const T *p, int64_t i) { return (double)p[i]; }

// Load a (rows x BK) panel of an operand whose element (r, k) is at p[r*sr + k*sk] into
// registers, one element per slot; out-of-range elements read as zero.  `kc` selects the mapping
// of lanes to elements so that consecutive lanes read consecutive addresses.
template <typename T, int ROWS, int BK>
__device__ __forceinline__ void load_panel(const T *p, int64_t sr, int64_t sk, int r0, int k0, int R, int K,
                                           double (&reg)[ROWS * BK / 256]) {
    constexpr int N = ROWS * BK / 256;
    const bool kc = (sk == 1);
#pragma unroll
    for (int s = 0; s < N; ++s) {
        int e = threadIdx.x + 256 * s;
        int r, k;
        if (kc) {
            r = e / BK;
            k = e % BK;
        } else {
            k = e / ROWS;
            r = e % ROWS;
        }
        const int gr = r0 + r, gk = k0 + k;
        // branch-free: an out-of-range slot reads element (0, 0) of the panel's operand (valid for
        // R, K >= 1) and is replaced by zero, so every slot's load is in flight at once
        const bool ok = gr < R && gk < K;
        const double v = ld(p, ok ? (int64_t)gr * sr + (int64_t)gk * sk : (int64_t)0);
        reg[s] = ok ? v : 0.0;
    }
}
// Range-checked panel walk: load_panel at every panel.
template <typename T, int ROWS, int BK>
struct CheckedPanels {
    const T *p;
    int64_t sr, sk;
    int R0, R, K;
    __device__ __forceinline__ void load(int k0, double (&reg)[ROWS * BK / 256]) const {
        load_panel<T, ROWS, BK>(p, sr, sk, R0, k0, R, K, reg);
    }
};

// Panel walk over an operand whose ROWS x K slab (rows R0.., all of the reduction) lies wholly in
// range, every byte of it within 2^31 of the slab's first element.  The lane -> element map of
// load_panel is affine in the slot (256 is a multiple of BK and of ROWS): slot s holds element
// (r + s dr, k + s dk), so each slot is one buffer load from a resource at the slab's origin, this
// lane's 32-bit byte offset (advanced by BK elements of the reduction per panel) and a uniform
// per-slot byte offset -- no per-slot index arithmetic or range test.
template <typename T, int ROWS, int BK>
struct InnerPanels {
    static_assert(256 % BK == 0 && 256 % ROWS == 0, "the slot map needs 256 to be a multiple of BK and ROWS");
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t voff0, kbytes, sbytes;
    __device__ __forceinline__ InnerPanels(const T *p, int64_t sr, int64_t sk, int R0) {
        const bool kc = (sk == 1);
        const int t = threadIdx.x;
        const int r = kc ? t / BK : t % ROWS, k = kc ? t % BK : t / ROWS;
        // raw buffer (stride 0), num_records in bytes; word 3 = 0x00020000 for the gfx9 family.  The
        // origin and the strides are the same in every lane: readfirstlane states it, so that the
        // resource and the slot offsets live in scalar registers.
        const uint64_t o = (uint64_t)(p + (int64_t)R0 * sr);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)o), hi = __builtin_amdgcn_readfirstlane((uint32_t)(o >> 32));
        rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), (short)0, 0x7fffffff, 0x00020000);
        voff0 = (uint32_t)(((int64_t)r * sr + (int64_t)k * sk) * (int64_t)sizeof(T));
        kbytes = __builtin_amdgcn_readfirstlane((uint32_t)(sk * (int64_t)sizeof(T)));
        sbytes = __builtin_amdgcn_readfirstlane((uint32_t)((kc ? (256 / BK) * sr : (256 / ROWS) * sk) * (int64_t)sizeof(T)));
    }
    // the slab fits the resource: rows R0 .. R0 + ROWS - 1 exist and the last element ends within 2^31 - 1 bytes
    static __device__ __forceinline__ bool fits(int64_t sr, int64_t sk, int R0, int R, int K) {
        return R0 + ROWS <= R && sr >= 0 && sk >= 0 &&
               ((int64_t)(ROWS - 1) * sr + (int64_t)(K - 1) * sk + 1) * (int64_t)sizeof(T) < ((int64_t)1 << 31);
    }
    __device__ __forceinline__ void load(int k0, double (&reg)[ROWS * BK / 256]) const {
        const uint32_t vo = voff0 + (uint32_t)k0 * kbytes;
#pragma unroll
        for (int s = 0; s < ROWS * BK / 256; ++s) {
            if constexpr (sizeof(T) == 8)
                reg[s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)vo, (int)(s * sbytes), 0));
            else
                reg[s] = (double)__builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)vo, (int)(s * sbytes), 0));
        }
    }
};

// ------------------------------------------------------------------------------------------------
// FP64 / FP32 kernels: 16x16x4 MFMA, LDS panels stored k-major [BK][ROWS + pad].
// MFMA 16x16x4 operand layout (per lane l of the wave): A value = A[i = l%16][k = l/16],
// B value = B[k = l/16][j = l%16].  Result registers v = 0..3 of lane l hold C[row][l%16] with
// row = 4*(l/16) + v for the FP32 form and row = l/16 + 4*v for the FP64 form.
// ------------------------------------------------------------------------------------------------
// IND: groups with device-side operands and coefficients (GemmIndirect; FP64).  A variant of its own, held
// to the plain kernel's 256 registers (two wavefronts per SIMD), which its epilogue would exceed by one.
// TRI: symmetric products (GemmGroup::tri), likewise.
template <typename TIN, typename TC, int BM, int BN, int BK, bool IND = false, bool TRI = false>
__global__ void __launch_bounds__(256, IND || TRI ? 2 : 1) k_gemm_fp(GemmArgs args) {
    int gi, b, tm, tn;
    if (!locate(args, gi, b, tm, tn)) return;
    const GemmGroup &g = args.g[gi];
    const int sp = b % g.splits;
    b /= g.splits;
    const int kb = sp * g.kchunk;
    const int K = min(g.K - kb, g.kchunk);
    const TIN *A = (const TIN *)g.A + b * g.sab + kb * g.sak;
    const TIN *B = (const TIN *)g.B + b * g.sbb + kb * g.sbk;
    TIN *C = (TIN *)g.C + b * g.scb + sp * g.scs;
    if constexpr (IND) {
        const int64_t t = b * g.ind.stride;
        if (g.ind.coef[t + 3] != 0.0) return;
        if (g.ind.a) A = g.ind.a[t] + kb * g.sak;
        if (g.ind.b) B = g.ind.b[t] + kb * g.sbk;
        if (g.ind.c && g.splits == 1) C = g.ind.c[t];
    }
    constexpr int PAD = 1;  // rows of BM + 1: lanes storing one k-column of a row-major panel hit distinct banks
    // FP32 tiles double-buffer their panels (one barrier per panel: 4 % faster on the 2048^3 FP32
    // contraction); the FP64 kernel keeps one buffer, which leaves it the registers for two waves
    // per SIMD
    constexpr int NBUF = sizeof(TC) == 4 ? 2 : 1;
    __shared__ TC As[NBUF][BK][BM + PAD];
    __shared__ TC Bs[NBUF][BK][BN + PAD];
    constexpr int NA = BM * BK / 256, NB = BN * BK / 256;
    constexpr int WM = BM / 2, WN = BN / 2, TI = WM / 16, TJ = WN / 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
    const int m0 = tm * BM, n0 = tn * BN;
    using acc_t = typename std::conditional<sizeof(TC) == 8, d4, f4>::type;
    acc_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    const bool akc = (g.sak == 1), bkc = (g.sbk == 1);
    // slot s of this lane holds panel element (r + s dr, k + s dk) and goes to Xs[k + s dk][r + s dr]
    const int t = threadIdx.x;
    const int lda0 = akc ? (t % BK) * (BM + PAD) + t / BK : (t / BM) * (BM + PAD) + t % BM;
    const int ldb0 = bkc ? (t % BK) * (BN + PAD) + t / BK : (t / BN) * (BN + PAD) + t % BN;
    const int lda_step = akc ? 256 / BK : (256 / BM) * (BM + PAD);
    const int ldb_step = bkc ? 256 / BK : (256 / BN) * (BN + PAD);

    // the matrix-core work on the panels in buffer `b`
    auto panel_mfma = [&](int b) {
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            TC af[TI], bf[TJ];
#pragma unroll
            for (int i = 0; i < TI; ++i) af[i] = As[b][kk + lane / 16][wm + 16 * i + lane % 16];
#pragma unroll
            for (int j = 0; j < TJ; ++j) bf[j] = Bs[b][kk + lane / 16][wn + 16 * j + lane % 16];
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j) {
                    if constexpr (sizeof(TC) == 8)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i], bf[j], acc[i][j], 0, 0, 0);
                    else
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bf[j], acc[i][j], 0, 0, 0);
                }
        }
    };
    auto mainloop = [&](const auto &la, const auto &lb) {
        double ra[NA], rb[NB];
        if constexpr (NBUF == 1) {
            if (K > 0) {
                la.load(0, ra);
                lb.load(0, rb);
            }
            for (int k0 = 0; k0 < K; k0 += BK) {
                __syncthreads();
#pragma unroll
                for (int s = 0; s < NA; ++s) (&As[0][0][0])[lda0 + s * lda_step] = (TC)ra[s];
#pragma unroll
                for (int s = 0; s < NB; ++s) (&Bs[0][0][0])[ldb0 + s * ldb_step] = (TC)rb[s];
                __syncthreads();
                if (k0 + BK < K) {  // prefetch the next panels while the matrix cores work
                    la.load(k0 + BK, ra);
                    lb.load(k0 + BK, rb);
                }
#pragma unroll
                for (int kk = 0; kk < BK; kk += 4) {
                    TC af[TI], bf[TJ];
#pragma unroll
                    for (int i = 0; i < TI; ++i) af[i] = As[0][kk + lane / 16][wm + 16 * i + lane % 16];
#pragma unroll
                    for (int j = 0; j < TJ; ++j) bf[j] = Bs[0][kk + lane / 16][wn + 16 * j + lane % 16];
#pragma unroll
                    for (int i = 0; i < TI; ++i)
#pragma unroll
                        for (int j = 0; j < TJ; ++j) {
                            if constexpr (sizeof(TC) == 8)
                                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i], bf[j], acc[i][j], 0, 0, 0);
                            else
                                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bf[j], acc[i][j], 0, 0, 0);
                        }
                }
            }
        } else {
            if (K <= 0) return;
            la.load(0, ra);
            lb.load(0, rb);
#pragma unroll
            for (int s = 0; s < NA; ++s) (&As[0][0][0])[lda0 + s * lda_step] = (TC)ra[s];
#pragma unroll
            for (int s = 0; s < NB; ++s) (&Bs[0][0][0])[ldb0 + s * ldb_step] = (TC)rb[s];
            if (BK < K) {
                la.load(BK, ra);
                lb.load(BK, rb);
            }
            __syncthreads();
            int cur = 0;
            for (int k0 = 0; k0 < K; k0 += BK) {
                // the next panels go to the other buffer (its last readers passed the barrier that
                // ended the previous panel), the ones after them into registers
                if (k0 + BK < K) {
#pragma unroll
                    for (int s = 0; s < NA; ++s) (&As[cur ^ 1][0][0])[lda0 + s * lda_step] = (TC)ra[s];
#pragma unroll
                    for (int s = 0; s < NB; ++s) (&Bs[cur ^ 1][0][0])[ldb0 + s * ldb_step] = (TC)rb[s];
                    if (k0 + 2 * BK < K) {
                        la.load(k0 + 2 * BK, ra);
                        lb.load(k0 + 2 * BK, rb);
                    }
                }
                panel_mfma(cur);
                __syncthreads();
                cur ^= 1;
            }
        }
    };
    // interior tiles with whole panels take the buffer-load walk, the others the range-checked one
    if (K % BK == 0 && InnerPanels<TIN, BM, BK>::fits(g.sam, g.sak, m0, g.M, K) &&
        InnerPanels<TIN, BN, BK>::fits(g.sbn, g.sbk, n0, g.N, K))
        mainloop(InnerPanels<TIN, BM, BK>(A, g.sam, g.sak, m0), InnerPanels<TIN, BN, BK>(B, g.sbn, g.sbk, n0));
    else
        mainloop(CheckedPanels<TIN, BM, BK>{A, g.sam, g.sak, m0, g.M, K},
                 CheckedPanels<TIN, BN, BK>{B, g.sbn, g.sbk, n0, g.N, K});
    double alpha = g.alpha, beta = g.beta, gamma = 0.0;
    const TIN *D = C;
    if constexpr (IND) {
        if (g.splits == 1) {  // (the partials of a split reduction are summed with these afterwards)
            const int64_t t = b * g.ind.stride;
            alpha = g.ind.coef[t];
            gamma = g.ind.coef[t + 1];
            beta = g.ind.coef[t + 2];
            if (gamma != 0.0) D = g.ind.d[t];
        }
    }
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = sizeof(TC) == 8 ? (lane / 16) + 4 * v : 4 * (lane / 16) + v;
                int r = m0 + wm + 16 * i + row;
                int c = n0 + wn + 16 * j + lane % 16;
                if (r < g.M && c < g.N) {
                    int64_t o = r * g.scm + c * g.scn;
                    double val = alpha * (double)acc[i][j][v];
                    if (beta != 0.0) val += beta * (double)C[o];
                    if constexpr (IND)
                        if (gamma != 0.0) val += gamma * (double)D[o];
                    C[o] = (TIN)val;
                    if constexpr (TRI)
                        if (tm != tn && g.splits == 1) C[c * g.scm + r * g.scn] = (TIN)val;
                }
            }
}

// ------------------------------------------------------------------------------------------------
// BF16 split-product kernel: 16x16x32 MFMA.  LDS panels stored row-major [ROWS][32 + pad] so that a
// lane's 8 consecutive k values are one 16-byte read.  Operand layout (lane l): A values
// A[i = l%16][k = 8*(l/16) + t], t = 0..7; B values B[k = 8*(l/16) + t][j = l%16]; the result layout
// is that of the 16x16x4 instructions.
// ------------------------------------------------------------------------------------------------
// SA / SB: BF16 terms each A / B element is split into (hi, mid, lo); the products of term t of A
// and term u of B with t + u < max(SA, SB) are accumulated, smallest first.
constexpr int kBfK = 32;             // reduction per panel: one MFMA
constexpr int kBfStride = kBfK + 8;  // 80-byte rows: the 16 rows of an operand read start in distinct banks
// k_gemm_pipe: a panel is four 16-byte slots a row, 2 FP64 or 4 FP32 k each; rows of 80 bytes, likewise
template <typename TC>
constexpr int kSlot = 16 / (int)sizeof(TC);
template <typename TC>
constexpr int kDepth = 4 * kSlot<TC>;
template <typename TC>
constexpr int kStride = 5 * kSlot<TC>;

// One operand's ROWS x BK panels in rows.  A lane's slot is V = BK / 4 consecutive k of one row, 16 bytes in
// LDS, kept in the operand's own type until it is stored.  Reduction-contiguous operands
// are read 16 bytes a lane (four lanes a row), row-contiguous ones one element a lane, 64 lanes on
// consecutive rows; panels that leave the operand, and origins or strides that 16-byte loads cannot
// take, are read element by element with a range check (out of range reads as zero).
template <typename T, int ROWS, int BK>
struct RowPanels {
    static constexpr int NS = ROWS / 64;  // slots per lane (256 lanes, 4 slots a row)
    static constexpr int V = BK / 4;
    typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
    const T *p;
    int64_t sr, sk;
    int R0, R, K;
    bool kc, wide, rows_in;
    T reg[NS][V];
    __device__ __forceinline__ RowPanels(const T *p_, int64_t sr_, int64_t sk_, int R0_, int R_, int K_)
        : p(p_), sr(sr_), sk(sk_), R0(R0_), R(R_), K(K_) {
        kc = sk == 1;
        wide = (((uint64_t)p) & 15) == 0 && (sr * (int64_t)sizeof(T)) % 16 == 0;
        rows_in = R0 + ROWS <= R;
    }
    __device__ __forceinline__ void at(int s, int &r, int &q) const {
        const int e = threadIdx.x + 256 * s;
        r = kc ? e / 4 : e % ROWS;
        q = kc ? e % 4 : e / ROWS;
    }
    __device__ __forceinline__ void load(int k0) {
        const bool inside = rows_in && k0 + BK <= K;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            int r, q;
            at(s, r, q);
            const int k = k0 + V * q;
            if (V * sizeof(T) >= 16 && inside && kc && wide) {
                const vec *src = (const vec *)(p + (int64_t)(R0 + r) * sr + k);
#pragma unroll
                for (int t = 0; t < V * (int)sizeof(T) / 16; ++t) {
                    const vec v = src[t];
#pragma unroll
                    for (int u = 0; u < 16 / (int)sizeof(T); ++u) reg[s][t * (16 / sizeof(T)) + u] = v[u];
                }
            } else if (inside) {
                const T *src = p + (int64_t)(R0 + r) * sr + (int64_t)k * sk;
#pragma unroll
                for (int t = 0; t < V; ++t) reg[s][t] = src[t * sk];
            } else {
#pragma unroll
                for (int t = 0; t < V; ++t) {
                    // branch-free: out of range reads element (0, 0), valid for R, K >= 1, and drops it
                    const bool ok = R0 + r < R && k + t < K;
                    const T v = p[ok ? (int64_t)(R0 + r) * sr + (int64_t)(k + t) * sk : (int64_t)0];
                    reg[s][t] = ok ? v : (T)0;
                }
            }
        }
    }
    // split into S terms; each rest x - hi is exact in T
    template <int S>
    __device__ __forceinline__ void store(__bf16 (&X)[S][ROWS][kBfStride]) const {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            int r, q;
            at(s, r, q);
            T x[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) x[t] = reg[s][t];
#pragma unroll
            for (int u = 0; u < S; ++u) {
                bf8 h;
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    h[t] = (__bf16)(float)x[t];
                    x[t] -= (T)(float)h[t];
                }
                *(bf8 *)&X[u][r][8 * q] = h;
            }
        }
    }
    template <typename TC>
    __device__ __forceinline__ void store(TC (&X)[ROWS][kStride<TC>]) const {
        static_assert(V == kSlot<TC>, "a slot is 16 bytes in LDS");
        typedef TC slot_t __attribute__((ext_vector_type(V)));
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            int r, q;
            at(s, r, q);
            slot_t h;
#pragma unroll
            for (int t = 0; t < V; ++t) h[t] = (TC)reg[s][t];
            *(slot_t *)&X[r][V * q] = h;
        }
    }
};

// Bounded by what surrounds the matrix instructions: with one element, widened to FP64, a lane and slot, two
// barriers a panel and 2-byte LDS stores, a 4096 x 256 x 256 product of five FP32 members (split A) took 45
// to 55 us, 15 at the rate of a large copy; with octets and two panel buffers (three terms have room for
// one) it takes 20 to 23.
template <typename TIN, int SA, int SB, int BM, int BN>
__global__ void __launch_bounds__(256, 2) k_gemm_bf16(GemmArgs args) {
    constexpr int NSPLIT = SA > SB ? SA : SB;
    constexpr int NBUF = NSPLIT > 2 ? 1 : 2;
    int gi, b, tm, tn;
    if (!locate(args, gi, b, tm, tn)) return;
    const GemmGroup &g = args.g[gi];
    const int sp = b % g.splits;
    b /= g.splits;
    const int kb = sp * g.kchunk;
    const int K = min(g.K - kb, g.kchunk);
    const TIN *A = (const TIN *)g.A + b * g.sab + kb * g.sak;
    const TIN *B = (const TIN *)g.B + b * g.sbb + kb * g.sbk;
    TIN *C = (TIN *)g.C + b * g.scb + sp * g.scs;
    __shared__ __attribute__((aligned(16))) __bf16 As[NBUF][SA][BM][kBfStride];
    __shared__ __attribute__((aligned(16))) __bf16 Bs[NBUF][SB][BN][kBfStride];
    constexpr int WM = BM / 2, WN = BN / 2, TI = WM / 16, TJ = WN / 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
    const int m0 = tm * BM, n0 = tn * BN;
    f4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = f4{0, 0, 0, 0};
    RowPanels<TIN, BM, kBfK> pa(A, g.sam, g.sak, m0, g.M, K);
    RowPanels<TIN, BN, kBfK> pb(B, g.sbn, g.sbk, n0, g.N, K);
    auto panel_mfma = [&](int buf) {
        bf8 af[SA][TI], bfr[SB][TJ];
#pragma unroll
        for (int t = 0; t < SA; ++t)
#pragma unroll
            for (int i = 0; i < TI; ++i) af[t][i] = *(const bf8 *)&As[buf][t][wm + 16 * i + lane % 16][8 * (lane / 16)];
#pragma unroll
        for (int t = 0; t < SB; ++t)
#pragma unroll
            for (int j = 0; j < TJ; ++j) bfr[t][j] = *(const bf8 *)&Bs[buf][t][wn + 16 * j + lane % 16][8 * (lane / 16)];
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                // small cross terms first, the hi*hi product last
                if constexpr (NSPLIT == 3) {
                    if constexpr (SA > 2) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[2][i], bfr[0][j], acc[i][j], 0, 0, 0);
                    if constexpr (SA > 1 && SB > 1) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[1][i], bfr[1][j], acc[i][j], 0, 0, 0);
                    if constexpr (SB > 2) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bfr[2][j], acc[i][j], 0, 0, 0);
                }
                if constexpr (NSPLIT >= 2) {
                    if constexpr (SA > 1) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[1][i], bfr[0][j], acc[i][j], 0, 0, 0);
                    if constexpr (SB > 1) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bfr[1][j], acc[i][j], 0, 0, 0);
                }
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bfr[0][j], acc[i][j], 0, 0, 0);
            }
    };
    if (K > 0) {
        pa.load(0);
        pb.load(0);
        int cur = 0;
        for (int k0 = 0; k0 < K; k0 += kBfK) {
            // two buffers: the one written here was last read before the barrier of the previous panel
            if constexpr (NBUF == 1) __syncthreads();
            pa.template store<SA>(As[cur]);
            pb.template store<SB>(Bs[cur]);
            if (k0 + kBfK < K) {  // the next panels are on their way while the matrix cores work
                pa.load(k0 + kBfK);
                pb.load(k0 + kBfK);
            }
            __syncthreads();
            panel_mfma(cur);
            if constexpr (NBUF == 2) cur ^= 1;
        }
    }
    const double alpha = g.alpha, beta = g.beta;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                int r = m0 + wm + 16 * i + 4 * (lane / 16) + v;
                int c = n0 + wn + 16 * j + lane % 16;
                if (r < g.M && c < g.N) {
                    int64_t o = r * g.scm + c * g.scn;
                    double val = alpha * (double)acc[i][j][v];
                    if (beta != 0.0) val += beta * (double)C[o];
                    C[o] = (TIN)val;
                }
            }
}

// RowPanels<T, ROWS, kDepth<TC>> where every panel lies inside the operand, within 2^31 bytes of the slab's first
// element: buffer loads from a scalar resource at the slab's origin, one 32-bit offset a lane and uniform
// offsets for the slots.  KC: reduction-contiguous on 16-byte boundaries; else row-contiguous (sr == 1).
template <typename T, typename TC, int ROWS, bool KC>
struct InnerRows {
    static constexpr int NS = ROWS / 64, V = kSlot<TC>;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t voff, kbytes, slot;
    int lds;
    T reg[NS][V];
    __device__ __forceinline__ InnerRows(const T *p, int64_t sr, int64_t sk, int R0) {
        const int t = threadIdx.x, r = KC ? t / 4 : t % ROWS, q = KC ? t % 4 : t / ROWS;
        const uint64_t o = (uint64_t)(p + (int64_t)R0 * sr);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)o), hi = __builtin_amdgcn_readfirstlane((uint32_t)(o >> 32));
        rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), (short)0, 0x7fffffff, 0x00020000);
        voff = (uint32_t)(((int64_t)r * sr + (int64_t)(V * q) * sk) * (int64_t)sizeof(T));
        kbytes = __builtin_amdgcn_readfirstlane((uint32_t)(sk * (int64_t)sizeof(T)));
        slot = __builtin_amdgcn_readfirstlane((uint32_t)((KC ? 64 * sr : V * (256 / ROWS) * sk) * (int64_t)sizeof(T)));
        lds = r * kStride<TC> + V * q;
    }
    static __device__ __forceinline__ bool fits(const T *p, int64_t sr, int64_t sk, int R0, int R, int K) {
        return (KC ? sk == 1 && (((uint64_t)p) & 15) == 0 && (sr * (int64_t)sizeof(T)) % 16 == 0 : sr == 1) && R0 + ROWS <= R &&
               sr >= 0 && sk >= 0 && ((int64_t)(ROWS - 1) * sr + (int64_t)(K - 1) * sk + 1) * (int64_t)sizeof(T) < ((int64_t)1 << 31);
    }
    __device__ __forceinline__ void load(int k0) {
        const uint32_t vo = voff + (uint32_t)k0 * kbytes;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if constexpr (KC && V * sizeof(T) >= 16) {
                typedef unsigned u4v __attribute__((ext_vector_type(4)));
#pragma unroll
                for (int h = 0; h < V * (int)sizeof(T) / 16; ++h) {
                    const u4v x = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(vo + 16 * h), (int)(s * slot), 0);
                    __builtin_memcpy(&reg[s][h * (16 / sizeof(T))], &x, 16);
                }
            } else {
#pragma unroll
                for (int t = 0; t < V; ++t) {
                    if constexpr (sizeof(T) == 8)
                        reg[s][t] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)vo, (int)(s * slot + t * kbytes), 0));
                    else
                        reg[s][t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)vo, (int)(s * slot + t * kbytes), 0));
                }
            }
        }
    }
    __device__ __forceinline__ void store(TC (&X)[ROWS][kStride<TC>]) const {
        typedef TC slot_t __attribute__((ext_vector_type(V)));
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            slot_t h;
#pragma unroll
            for (int t = 0; t < V; ++t) h[t] = (TC)reg[s][t];
            *(slot_t *)(&X[0][0] + lds + s * (KC ? 64 * kStride<TC> : V * (256 / ROWS))) = h;
        }
    }
};

// Products with unbroken matrix work, in FP64, and in FP32 on FP32 operands: 16x16x4 MFMA on panels in rows, two
// LDS buffers, one barrier a panel of eight (FP32: sixteen).  Lane l holds the slot of k = V (l / 16) .. + V - 1
// of its row, one 16-byte read, and the s-th of a panel's V instructions per tile multiplies the s-th of them:
// the same k in both operands, which is all that the sum asks for.  What fills LDS and registers for the next
// panels is placed between the matrix instructions (`panel`).  Against k_gemm_fp (panels of 16 stored k by k,
// LDS waits in the open and, in FP64, two barriers around one buffer a panel), TFLOP/s on N(0,1) entries, FP64:
// 8192^3 67.5 -> 75.3, two products of 2048^3 61 to 65 -> 71, 32 of 2048 x 128 x 2048 58 to 61 -> 65, nominal
// peak 78.6 (torch's products beside it 69 to 73 on the square sizes); FP32: 8192^3 109 -> 149, two of 2048^3
// 110 -> 140, peak 157.  Launches that leave most of a compute unit idle wait for memory more often with the
// shorter panels (59 products of 640 x 128 x 640 took 835 us and not 780), and the range finder's epilogue would
// spill: those stay with k_gemm_fp, and the autotuner times both for the others.  So does FP32 arithmetic on FP64
// operands, bound by their conversion (105 to 112 against 110 to 113).  TRI: symmetric products.
template <typename TIN, typename TC, int BM, int BN, bool TRI = false>
__global__ void __launch_bounds__(256, 2) k_gemm_pipe(GemmArgs args) {
    int gi, b, tm, tn;
    if (!locate(args, gi, b, tm, tn)) return;
    const GemmGroup &g = args.g[gi];
    const int sp = b % g.splits;
    b /= g.splits;
    const int kb = sp * g.kchunk;
    const int K = min(g.K - kb, g.kchunk);
    const TIN *A = (const TIN *)g.A + b * g.sab + kb * g.sak;
    const TIN *B = (const TIN *)g.B + b * g.sbb + kb * g.sbk;
    TIN *C = (TIN *)g.C + b * g.scb + sp * g.scs;
    constexpr int V = kSlot<TC>, DEPTH = kDepth<TC>;
    __shared__ __attribute__((aligned(16))) TC As[2][BM][kStride<TC>];
    __shared__ __attribute__((aligned(16))) TC Bs[2][BN][kStride<TC>];
    constexpr int WM = BM / 2, WN = BN / 2, TI = WM / 16, TJ = WN / 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
    const int m0 = tm * BM, n0 = tn * BN;
    using acc_t = typename std::conditional<sizeof(TC) == 8, d4, f4>::type;
    acc_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    typedef TC slot_t __attribute__((ext_vector_type(V)));
    struct Frag {
        slot_t a[TI], b[TJ];
    };
    auto fetch = [&](int buf, Frag &f) {
#pragma unroll
        for (int i = 0; i < TI; ++i) f.a[i] = *(const slot_t *)&As[buf][wm + 16 * i + lane % 16][V * (lane / 16)];
#pragma unroll
        for (int j = 0; j < TJ; ++j) f.b[j] = *(const slot_t *)&Bs[buf][wn + 16 * j + lane % 16][V * (lane / 16)];
    };
    auto multiply = [&](const Frag &f, int half) {  // V / 2 of a panel's V instructions per tile
#pragma unroll
        for (int s = half * (V / 2); s < (half + 1) * (V / 2); ++s)
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j) {
                    if constexpr (sizeof(TC) == 8)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[i][s], f.b[j][s], acc[i][j], 0, 0, 0);
                    else
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.a[i][s], f.b[j][s], acc[i][j], 0, 0, 0);
                }
    };
    // One panel, its operands in `f`: the next panel's go to LDS and the one after that is loaded while the
    // first half of the instructions runs, and after the barrier the next panel's operands are read into
    // `next` under the second half; the groups put this order between the instructions.  (Buffer `to` was last
    // read before the barrier of the panel before.)
    auto panel = [&](auto &pa, auto &pb, const Frag &f, Frag &next, int to, int k2, auto has1, auto has2) {
        if constexpr (decltype(has1)::value) {
            pa.store(As[to]);
            pb.store(Bs[to]);
        }
        if constexpr (decltype(has2)::value) {
            pa.load(k2);
            pb.load(k2);
        }
        multiply(f, 0);
        if constexpr (decltype(has2)::value) {
#pragma unroll
            for (int t = 0; t < TI * TJ; ++t) {
                __builtin_amdgcn_sched_group_barrier(0x008, V / 2, 0);  // matrix
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // load
                __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // vector
            }
        }
        if constexpr (decltype(has1)::value) {
            __syncthreads();
            fetch(to, next);
        }
        multiply(f, 1);
        if constexpr (decltype(has1)::value) {
#pragma unroll
            for (int t = 0; t < TI + TJ; ++t) {
                __builtin_amdgcn_sched_group_barrier(0x008, V / 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
            }
        }
    };
    auto mainloop = [&](auto &&pa, auto &&pb) {
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        if (K <= 0) return;
        pa.load(0);
        pb.load(0);
        pa.store(As[0]);
        pb.store(Bs[0]);
        if (K > DEPTH) {
            pa.load(DEPTH);
            pb.load(DEPTH);
        }
        __syncthreads();
        Frag f0, f1;
        fetch(0, f0);
        int k0 = 0;
        for (; k0 + 3 * DEPTH < K; k0 += 2 * DEPTH) {  // two panels a turn: neither set of operands is copied
            panel(pa, pb, f0, f1, 1, k0 + 2 * DEPTH, yes, yes);
            panel(pa, pb, f1, f0, 0, k0 + 3 * DEPTH, yes, yes);
        }
        // one to three panels are left, the first of them in f0
        if (k0 + 2 * DEPTH < K) {
            panel(pa, pb, f0, f1, 1, k0 + 2 * DEPTH, yes, yes);
            panel(pa, pb, f1, f0, 0, 0, yes, no);
            panel(pa, pb, f0, f1, 1, 0, no, no);
        } else if (k0 + DEPTH < K) {
            panel(pa, pb, f0, f1, 1, 0, yes, no);
            panel(pa, pb, f1, f0, 0, 0, no, no);
        } else {
            panel(pa, pb, f0, f1, 1, 0, no, no);
        }
    };
    const bool whole = K % DEPTH == 0;
    const bool akc = g.sak == 1, bkc = g.sbk == 1;
    const bool fast_a = whole && (akc ? InnerRows<TIN, TC, BM, true>::fits(A, g.sam, g.sak, m0, g.M, K)
                                      : InnerRows<TIN, TC, BM, false>::fits(A, g.sam, g.sak, m0, g.M, K));
    const bool fast_b = whole && (bkc ? InnerRows<TIN, TC, BN, true>::fits(B, g.sbn, g.sbk, n0, g.N, K)
                                      : InnerRows<TIN, TC, BN, false>::fits(B, g.sbn, g.sbk, n0, g.N, K));
    if (fast_a && fast_b && akc && !bkc)
        mainloop(InnerRows<TIN, TC, BM, true>(A, g.sam, g.sak, m0), InnerRows<TIN, TC, BN, false>(B, g.sbn, g.sbk, n0));
    else if (fast_a && fast_b && !akc && !bkc)
        mainloop(InnerRows<TIN, TC, BM, false>(A, g.sam, g.sak, m0), InnerRows<TIN, TC, BN, false>(B, g.sbn, g.sbk, n0));
    else if (fast_a && fast_b && bkc && akc)
        mainloop(InnerRows<TIN, TC, BM, true>(A, g.sam, g.sak, m0), InnerRows<TIN, TC, BN, true>(B, g.sbn, g.sbk, n0));
    else
        mainloop(RowPanels<TIN, BM, DEPTH>(A, g.sam, g.sak, m0, g.M, K), RowPanels<TIN, BN, DEPTH>(B, g.sbn, g.sbk, n0, g.N, K));
    const double alpha = g.alpha, beta = g.beta;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = sizeof(TC) == 8 ? (lane / 16) + 4 * v : 4 * (lane / 16) + v;
                int r = m0 + wm + 16 * i + row;
                int c = n0 + wn + 16 * j + lane % 16;
                if (r < g.M && c < g.N) {
                    int64_t o = r * g.scm + c * g.scn;
                    double val = alpha * (double)acc[i][j][v];
                    if (beta != 0.0) val += beta * (double)C[o];
                    C[o] = (TIN)val;
                    if constexpr (TRI)
                        if (tm != tn && g.splits == 1) C[c * g.scm + r * g.scn] = (TIN)val;
                }
            }
}

// Lane-layout self-test: A[i][0] = 1, A[i][1] = i, B[0][j] = j + 1, B[1][j] = 16 (other k zero), so
// D[i][j] = 16 i + j + 1.  Each lane feeds the operand elements the GEMM kernels assume it holds and
// stores its four result registers.  One wavefront; writes exactly 768 doubles.
__device__ __forceinline__ double probe_a(int i, int k) { return k == 0 ? 1.0 : (k == 1 ? (double)i : 0.0); }
__device__ __forceinline__ double probe_b(int k, int j) { return k == 0 ? (double)(j + 1) : (k == 1 ? 16.0 : 0.0); }

__global__ void __launch_bounds__(64) k_mfma_selftest(double *out) {
    const int l = threadIdx.x;
    if (l >= 64) return;
    const int r = l % 16, q = l / 16;
    d4 a64 = {0, 0, 0, 0};
    a64 = __builtin_amdgcn_mfma_f64_16x16x4f64(probe_a(r, q), probe_b(q, r), a64, 0, 0, 0);
    f4 a32 = {0, 0, 0, 0};
    a32 = __builtin_amdgcn_mfma_f32_16x16x4f32((float)probe_a(r, q), (float)probe_b(q, r), a32, 0, 0, 0);
    bf8 av, bv;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        av[t] = (__bf16)(float)probe_a(r, 8 * q + t);
        bv[t] = (__bf16)(float)probe_b(8 * q + t, r);
    }
    f4 ab = {0, 0, 0, 0};
    ab = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, ab, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        out[4 * l + v] = a64[v];
        out[256 + 4 * l + v] = (double)a32[v];
        out[512 + 4 * l + v] = (double)ab[v];
    }
}

// C[b](r, c) = alpha * sum_sp W[b][sp](r, c) + beta * C[b](r, c) over the split partials W
// (batch x splits consecutive M x N matrices), in a fixed order; an indirect group's operands and
// coefficients come from its tables.
template <typename T>
__global__ void k_split_sum(const T *__restrict__ W, int splits, int M, int N, int batch, T *C, int64_t scm,
                            int64_t scn, int64_t scb, double alpha, double beta, GemmIndirect ind, int tri) {
    const int64_t MN = (int64_t)M * N, total = MN * batch;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = i / MN, e = i - b * MN;
        const int64_t r = e / N, c = e - r * N;
        const T *w = W + b * splits * MN + e;
        double acc = 0.0;
        if constexpr (sizeof(T) == 8) {
            if (ind.coef) {
                const int64_t t = b * ind.stride, o = r * scm + c * scn;
                if (ind.coef[t + 3] != 0.0) continue;
                for (int sp = 0; sp < splits; ++sp) acc += (double)w[sp * MN];
                T *Cb = ind.c ? ind.c[t] : C + b * scb;
                double v = ind.coef[t] * acc;
                if (ind.coef[t + 2] != 0.0) v += ind.coef[t + 2] * Cb[o];
                if (ind.coef[t + 1] != 0.0) v += ind.coef[t + 1] * ind.d[t][o];
                Cb[o] = v;
                continue;
            }
        }
        if (tri && r / tri > c / tri) continue;  // a tile (of tri rows) that was not computed
        for (int sp = 0; sp < splits; ++sp) acc += (double)w[sp * MN];
        const int64_t o = b * scb + r * scm + c * scn;
        double v = alpha * acc;
        if (beta != 0.0) v += beta * (double)C[o];
        C[o] = (T)v;
        if (tri && r / tri < c / tri) C[b * scb + c * scm + r * scn] = (T)v;
    }
}

// Split-K workspace: one grow-only buffer per device, under g_ws_mu from a launch's look-up to its last use.
// Launches on one stream are ordered; a launch on another stream first waits for the event recorded after
// the buffer's last use.  Inside a SplitScope the record is left to the scope's end or to the first other
// stream, whose thread records it behind all that the last stream has been given by then.
struct SplitWs {
    void *p = nullptr;
    size_t bytes = 0;
    hipStream_t last = nullptr;
    hipEvent_t done = nullptr;
    bool used = false;
    const SplitScope *pending = nullptr;  // the scope whose use the event does not cover yet
};
static std::mutex g_ws_mu;
static std::map<int, SplitWs> g_ws;
static thread_local const SplitScope *t_scope = nullptr;  // this thread's open scope

static int split_done(SplitWs &w) {
    w.pending = nullptr;
    GTN_CHECK_HIP(hipEventRecord(w.done, w.last));
    return GTN_OK;
}

SplitScope::SplitScope() : outer_(t_scope != nullptr) {
    if (!outer_) t_scope = this;
}

int SplitScope::finish() {
    if (!open_) return GTN_OK;
    open_ = false;
    if (outer_) return GTN_OK;
    t_scope = nullptr;
    int rc = GTN_OK;
    std::lock_guard<std::mutex> l(g_ws_mu);
    for (auto &kv : g_ws)
        if (kv.second.pending == this) {
            const int r = split_done(kv.second);
            if (r) rc = r;
        }
    return rc;
}

static std::vector<void *> g_ws_retired;  // outgrown workspaces a graph may still hold

static int split_workspace(SplitWs &w, size_t bytes, hipStream_t s) {
    if (w.used && w.last != s) {
        if (w.pending) {
            int rc = split_done(w);
            if (rc) return rc;
        }
        GTN_CHECK_HIP(hipStreamWaitEvent(s, w.done, 0));
    }
    if (w.bytes < bytes) {
        if (w.p) {
            if (graphs_alive() || capture_open()) {
                g_ws_retired.push_back(w.p);  // kept: a captured graph may address it
            } else {
                GTN_CHECK_HIP(hipDeviceSynchronize());
                GTN_CHECK_HIP(hipFree(w.p));
            }
            w.p = nullptr;
            w.bytes = 0;
        }
        GTN_CHECK_HIP(hipMalloc(&w.p, bytes));
        w.bytes = bytes;
    }
    if (!w.done) GTN_CHECK_HIP(hipEventCreateWithFlags(&w.done, hipEventDisableTiming));
    return GTN_OK;
}

// tile: 64 (64 x 64 tiles) or 128 (128 x 128 tiles; each of the 4 wavefronts owns 64 x 64)
template <typename TIN>
static int launch_gemm(GemmArgs &a, int precision, int tile, bool pipe, hipStream_t s) {
    int total = a.tile_start[a.n_groups];
    if (total == 0) return GTN_OK;
    int grid = (total + 7) / 8 * 8;
    const bool big = tile == 128;
    switch (precision) {
        case GTN_PREC_F64:
            if (pipe && !a.g[0].ind.coef) {
                if constexpr (sizeof(TIN) == 8) {
                    if (a.g[0].tri) {
                        if (big)
                            hipLaunchKernelGGL((k_gemm_pipe<TIN, double, 128, 128, true>), dim3(grid), dim3(256), 0, s, a);
                        else
                            hipLaunchKernelGGL((k_gemm_pipe<TIN, double, 64, 64, true>), dim3(grid), dim3(256), 0, s, a);
                        break;
                    }
                }
                if (big)
                    hipLaunchKernelGGL((k_gemm_pipe<TIN, double, 128, 128>), dim3(grid), dim3(256), 0, s, a);
                else
                    hipLaunchKernelGGL((k_gemm_pipe<TIN, double, 64, 64>), dim3(grid), dim3(256), 0, s, a);
                break;
            }
            if constexpr (sizeof(TIN) == 8) {
                if (a.g[0].tri) {
                    if (big)
                        hipLaunchKernelGGL((k_gemm_fp<TIN, double, 128, 128, 16, false, true>), dim3(grid), dim3(256), 0, s, a);
                    else
                        hipLaunchKernelGGL((k_gemm_fp<TIN, double, 64, 64, 16, false, true>), dim3(grid), dim3(256), 0, s, a);
                    break;
                }
                if (a.g[0].ind.coef) {
                    if (big)
                        hipLaunchKernelGGL((k_gemm_fp<TIN, double, 128, 128, 16, true>), dim3(grid), dim3(256), 0, s, a);
                    else
                        hipLaunchKernelGGL((k_gemm_fp<TIN, double, 64, 64, 16, true>), dim3(grid), dim3(256), 0, s, a);
                    break;
                }
            }
            if (big)
                hipLaunchKernelGGL((k_gemm_fp<TIN, double, 128, 128, 16>), dim3(grid), dim3(256), 0, s, a);
            else
                hipLaunchKernelGGL((k_gemm_fp<TIN, double, 64, 64, 16>), dim3(grid), dim3(256), 0, s, a);
            break;
        case GTN_PREC_F32:
            if constexpr (sizeof(TIN) == 4) {
                if (pipe) {
                    if (big)
                        hipLaunchKernelGGL((k_gemm_pipe<TIN, float, 128, 128>), dim3(grid), dim3(256), 0, s, a);
                    else
                        hipLaunchKernelGGL((k_gemm_pipe<TIN, float, 64, 64>), dim3(grid), dim3(256), 0, s, a);
                    break;
                }
            }
            if (big)
                hipLaunchKernelGGL((k_gemm_fp<TIN, float, 128, 128, 16>), dim3(grid), dim3(256), 0, s, a);
            else
                hipLaunchKernelGGL((k_gemm_fp<TIN, float, 64, 64, 16>), dim3(grid), dim3(256), 0, s, a);
            break;
        case GTN_PREC_BF16X3:
            if (big)
                hipLaunchKernelGGL((k_gemm_bf16<TIN, 2, 2, 128, 128>), dim3(grid), dim3(256), 0, s, a);
            else
                hipLaunchKernelGGL((k_gemm_bf16<TIN, 2, 2, 64, 64>), dim3(grid), dim3(256), 0, s, a);
            break;
        case GTN_PREC_BF16X6:
            if (big)
                hipLaunchKernelGGL((k_gemm_bf16<TIN, 3, 3, 128, 128>), dim3(grid), dim3(256), 0, s, a);
            else
                hipLaunchKernelGGL((k_gemm_bf16<TIN, 3, 3, 64, 64>), dim3(grid), dim3(256), 0, s, a);
            break;
        case GTN_PREC_BF16:
            if (big)
                hipLaunchKernelGGL((k_gemm_bf16<TIN, 1, 1, 128, 128>), dim3(grid), dim3(256), 0, s, a);
            else
                hipLaunchKernelGGL((k_gemm_bf16<TIN, 1, 1, 64, 64>), dim3(grid), dim3(256), 0, s, a);
            break;
        case GTN_PREC_BF16_SPLIT_A:
            if (big)
                hipLaunchKernelGGL((k_gemm_bf16<TIN, 2, 1, 128, 128>), dim3(grid), dim3(256), 0, s, a);
            else
                hipLaunchKernelGGL((k_gemm_bf16<TIN, 2, 1, 64, 64>), dim3(grid), dim3(256), 0, s, a);
            break;
        default: set_error("gtn_gemm_grouped: unknown precision %d", precision); return GTN_ENOTSUP;
    }
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

// 128 x 128 tiles when every group is at least 128 x 128 and the launch still has a tile for every
// compute unit; 64 x 64 otherwise.  GTN_GEMM_TILE=64|128 in the environment forces a size (128 only
// where every group is at least 128 x 128) for tuning and tests.
static int pick_tile(const gtn_gemm_desc *groups, int n, bool tri) {
    static int forced = -1;
    if (forced < 0) {
        const char *e = getenv("GTN_GEMM_TILE");
        forced = e ? atoi(e) : 0;
    }
    int64_t t128 = 0;
    for (int i = 0; i < n; ++i) {
        const gtn_gemm_desc &d = groups[i];
        if (d.M == 0 || d.N == 0 || d.batch == 0) continue;
        if (d.M < 128 || d.N < 128) return 64;
        const int64_t tn = (d.N + 127) / 128;
        t128 += (tri ? tn * (tn + 1) / 2 : ((d.M + 127) / 128) * tn) * d.batch;
    }
    if (forced == 64 || forced == 128) return forced;
    return t128 >= 256 ? 128 : 64;
}

// GTN_GEMM_SPLIT=0 in the environment turns the split reduction off; GTN_GEMM_SPLIT=n > 1 sets the
// workgroup count a split launch aims for (default 1024) (tuning and tests).
static int split_target() {
    static int target = -1;
    if (target < 0) {
        const char *e = getenv("GTN_GEMM_SPLIT");
        const int v = e ? atoi(e) : 1024;
        target = v == 0 ? 0 : (v > 1 ? v : 1024);
    }
    return target;
}

}  // namespace gtn

using namespace gtn;

// Split-reduction scratch of gtn_gemm_grouped_noalloc: one fixed array per device, held for the life
// of the process.  In host code `scratch` only names the symbol; its device address on the current
// device comes from hipGetSymbolAddress (scratch_ptr below) and is what kernels are given.
constexpr int64_t kNoAllocScratchBytes = 64ll << 20;
static __device__ __align__(256) char scratch[kNoAllocScratchBytes];
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices];

// device address of `scratch` on the current device, looked up once per device
static int scratch_ptr(void **out) {
    int dev;
    GTN_CHECK_HIP(hipGetDevice(&dev));
    GTN_REQUIRE(dev >= 0 && dev < kMaxDevices, "gtn_gemm_grouped_noalloc: device index %d out of range", dev);
    std::lock_guard<std::mutex> l(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error("gtn_gemm_grouped_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                      hipGetErrorString(e));
            return GTN_EDEVICE;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return GTN_OK;
}

// The grouped GEMM.  fixed_ws == nullptr: split-reduction partials go to the library's per-device
// workspace (allocated and grown here).  Otherwise they go to fixed_ws (fixed_bytes long) and a
// split plan that needs more is an error; nothing is allocated.
// tile <= 0 / target < 0: the heuristics (pick_tile, split_target)
static int gemm_grouped_impl(const gtn_gemm_desc *groups, int n_groups, int dtype, int precision, void *stream,
                             void *fixed_ws, int64_t fixed_bytes, const char *name, int tile_cfg = 0,
                             int target_cfg = -1, const GemmIndirect *ind = nullptr, bool tri = false, int pipe_cfg = -1) {
    GTN_REQUIRE(n_groups >= 0 && (n_groups == 0 || groups), "%s: bad groups", name);
    GTN_REQUIRE(dtype == GTN_F64 || dtype == GTN_F32, "gtn_gemm_grouped: dtype must be F64 or F32");
    const int tile = tile_cfg > 0 ? tile_cfg : pick_tile(groups, n_groups, tri);
    const int BM = tile, BN = tile;
    const bool pipe = pipe_cfg >= 0 ? pipe_cfg : tile == 128;  // untuned: launches that fill the device (pick_tile)
    hipStream_t s = as_stream(stream);
    for (int base = 0; base < n_groups; base += kMaxGroups) {
        GemmArgs a;
        memset(&a, 0, sizeof(a));
        int n = n_groups - base < kMaxGroups ? n_groups - base : kMaxGroups;
        int tiles = 0;
        int used = 0;
        for (int i = 0; i < n; ++i) {
            const gtn_gemm_desc &d = groups[base + i];
            GTN_REQUIRE(d.M >= 0 && d.N >= 0 && d.K >= 0 && d.batch >= 0, "gtn_gemm_grouped: negative size");
            GTN_REQUIRE(d.M < (1 << 30) && d.N < (1 << 30) && d.K < (1 << 30), "gtn_gemm_grouped: size too large");
            GTN_REQUIRE(d.sak == 1 || d.sam == 1 || d.M <= 1 || d.K <= 1, "gtn_gemm_grouped: A needs a unit stride");
            GTN_REQUIRE(d.sbk == 1 || d.sbn == 1 || d.N <= 1 || d.K <= 1, "gtn_gemm_grouped: B needs a unit stride");
            if (d.M == 0 || d.N == 0 || d.batch == 0) continue;
            GTN_REQUIRE(d.A && d.B && d.C, "gtn_gemm_grouped: null operand");
            GemmGroup &g = a.g[used];
            g.A = d.A;
            g.B = d.B;
            g.C = d.C;
            g.M = (int32_t)d.M;
            g.N = (int32_t)d.N;
            g.K = (int32_t)d.K;
            g.batch = (int32_t)d.batch;
            g.tiles_m = (int32_t)((d.M + BM - 1) / BM);
            g.tiles_n = (int32_t)((d.N + BN - 1) / BN);
            // a unit stride on a length-1 dimension is ambiguous; normalise so the loader picks
            // the contiguous mapping
            g.sam = d.sam;
            g.sak = d.sak;
            if (d.K <= 1) g.sak = 1;
            g.sbk = d.sbk;
            g.sbn = d.sbn;
            if (d.K <= 1) g.sbk = 1;
            g.scm = d.scm;
            g.scn = d.scn;
            g.sab = d.sab;
            g.sbb = d.sbb;
            g.scb = d.scb;
            g.alpha = d.alpha;
            g.beta = d.beta;
            if (ind) g.ind = ind[base + i];
            g.tri = tri;
            g.splits = 1;
            g.kchunk = g.K;
            g.scs = 0;
            a.tile_start[used] = tiles;
            int64_t t = (tri ? (int64_t)g.tiles_n * (g.tiles_n + 1) / 2 : (int64_t)g.tiles_m * g.tiles_n) * g.batch;
            GTN_REQUIRE(tiles + t < (1ll << 31), "gtn_gemm_grouped: too many tiles");
            tiles += (int)t;
            ++used;
        }
        a.n_groups = used;
        a.tile_start[used] = tiles;
        if (used == 0) continue;
        if (dry_run()) {
            const int es = dtype == GTN_F64 ? 8 : 4;
            for (int i = 0; i < used; ++i) {
                const GemmGroup &q = a.g[i];
                int64_t lastb = q.batch - 1;
                int64_t ea = q.K > 0 ? lastb * q.sab + (int64_t)(q.M - 1) * q.sam + (int64_t)(q.K - 1) * q.sak + 1 : 0;
                int64_t eb = q.K > 0 ? lastb * q.sbb + (int64_t)(q.K - 1) * q.sbk + (int64_t)(q.N - 1) * q.sbn + 1 : 0;
                int64_t ec = lastb * q.scb + (int64_t)(q.M - 1) * q.scm + (int64_t)(q.N - 1) * q.scn + 1;
                GTN_RANGE(q.A, ea * es, "gemm A");
                GTN_RANGE(q.B, eb * es, "gemm B");
                GTN_RANGE(q.C, ec * es, "gemm C");
            }
            continue;
        }
        // Too few tiles to give every compute unit two workgroups: cut long reductions into chunks
        // (partials to the workspace, summed in a fixed order afterwards) until the launch has about
        // four workgroups per compute unit (the split target).  A chunk keeps at least 256 of the
        // reduction.
        const int es = dtype == GTN_F64 ? 8 : 4;
        std::vector<GemmGroup> orig;
        std::unique_lock<std::mutex> lk(g_ws_mu, std::defer_lock);
        SplitWs *ws = nullptr;
        const int target = target_cfg >= 0 ? target_cfg : split_target();
        if (tiles < 512 && target > 0 && tiles * 2 <= target) {
            int S = 1;
            while (tiles * S < target && S < 16) S *= 2;
            int64_t need = 0;
            int splitting = 0;
            for (int i = 0; i < used; ++i) {
                GemmGroup &g = a.g[i];
                int Sg = S;
                while (Sg > 1 && g.K / Sg < 256) Sg /= 2;
                if (Sg > 1) {
                    const int chunk = (g.K / Sg + 31) / 32 * 32;
                    Sg = (g.K + chunk - 1) / chunk;
                    g.splits = Sg;
                    g.kchunk = chunk;
                    need += (int64_t)Sg * g.batch * g.M * g.N;
                    ++splitting;
                }
            }
            if (splitting) {
                char *base_ws;
                if (fixed_ws) {
                    if (need * es > fixed_bytes) {
                        set_error("%s: the split reduction needs %lld bytes of scratch, above its maximum of %lld bytes",
                                  name, (long long)(need * es), (long long)fixed_bytes);
                        return GTN_ENOMEM;
                    }
                    base_ws = (char *)fixed_ws;
                } else {
                    int dev;
                    GTN_CHECK_HIP(hipGetDevice(&dev));
                    lk.lock();
                    ws = &g_ws[dev];
                    int rc = split_workspace(*ws, (size_t)need * es, s);
                    if (rc) return rc;
                    base_ws = (char *)ws->p;
                }
                orig.assign(a.g, a.g + used);
                int64_t off = 0;
                tiles = 0;
                for (int i = 0; i < used; ++i) {
                    GemmGroup &g = a.g[i];
                    a.tile_start[i] = tiles;
                    if (g.splits > 1) {
                        g.C = base_ws + off * es;
                        g.scm = g.N;
                        g.scn = 1;
                        g.scs = (int64_t)g.M * g.N;
                        g.scb = g.scs * g.splits;
                        g.alpha = 1.0;
                        g.beta = 0.0;
                        off += g.scb * g.batch;
                    }
                    tiles += (tri ? g.tiles_n * (g.tiles_n + 1) / 2 : g.tiles_m * g.tiles_n) * g.batch * g.splits;
                }
                a.tile_start[used] = tiles;
            }
        }
        int rc = dtype == GTN_F64 ? launch_gemm<double>(a, precision, tile, pipe, s) : launch_gemm<float>(a, precision, tile, pipe, s);
        if (rc) return rc;
        if (!orig.empty()) {
            for (int i = 0; i < used; ++i) {
                const GemmGroup &g = a.g[i], &o = orig[i];
                if (g.splits == 1) continue;
                const dim3 grid(grid_for((int64_t)g.M * g.N * g.batch, 256, 4096)), blk(256);
                if (dtype == GTN_F64)
                    hipLaunchKernelGGL(k_split_sum<double>, grid, blk, 0, s, (const double *)g.C, g.splits, g.M, g.N,
                                       g.batch, (double *)o.C, o.scm, o.scn, o.scb, o.alpha, o.beta, o.ind,
                                       o.tri ? BM : 0);
                else
                    hipLaunchKernelGGL(k_split_sum<float>, grid, blk, 0, s, (const float *)g.C, g.splits, g.M, g.N,
                                       g.batch, (float *)o.C, o.scm, o.scn, o.scb, o.alpha, o.beta, o.ind,
                                       o.tri ? BM : 0);
                GTN_CHECK_LAUNCH();
            }
            if (ws) {
                ws->last = s;
                ws->used = true;
                if (t_scope) {
                    ws->pending = t_scope;
                } else {
                    int rcd = split_done(*ws);
                    if (rcd) return rcd;
                }
            }
        }
    }
    return GTN_OK;
}

// ---- autotuner: launch configuration per call signature -------------------------------------
// Candidates: tile 64 or 128 (128 only where every group is at least 128 x 128) times split-K
// target 0 (no split), 512, 1024 or 2048 workgroups, on k_gemm_fp, and then, where there is one,
// k_gemm_pipe in both tiles at the split found best and the usual one.  The first eager call of a signature (element
// type, precision, and per group M, N, K, batch and operand layouts) times every candidate with HIP
// events (best of kTuneReps launches each) on its own operands and keeps the fastest; calls made while
// the stream is capturing a graph, and calls with beta != 0 (whose output a trial would change), use
// the tuned configuration when there is one and the heuristics otherwise.
struct TuneCfg {
    int tile, target;
    float ms, ms_default;
    int pipe;
};
static std::mutex g_tune_mu;
static std::map<std::string, TuneCfg> g_tuned;
static int g_autotune = -1;
constexpr int kTuneReps = 3;

static bool autotune_on() {
    if (g_autotune < 0) {
        const char *e = getenv("GTN_AUTOTUNE");
        g_autotune = e ? (atoi(e) != 0) : 1;
    }
    return g_autotune == 1;
}

enum { kPlain = 0, kTri = 1, kIndirect = 2 };  // kinds of launches, tuned apart
static std::string tune_key(const gtn_gemm_desc *g, int n, int dtype, int prec, int dev, int kind) {
    std::string k;
    auto put = [&](int64_t v) { k.append((const char *)&v, sizeof(v)); };
    put(dev);
    put(dtype);
    put(prec);
    put(n);
    for (int i = 0; i < n; ++i) {
        put(g[i].M);
        put(g[i].N);
        put(g[i].K);
        put(g[i].batch);
        put((g[i].sak == 1) | ((g[i].sbk == 1) << 1) | ((g[i].scn == 1) << 2) | (kind << 3));
    }
    return k;
}

static int time_cfg(const gtn_gemm_desc *groups, int n, int dtype, int prec, hipStream_t s, int tile, int target,
                    hipEvent_t e0, hipEvent_t e1, float *best, bool tri, int pipe) {
    *best = 1e30f;
    for (int r = 0; r < kTuneReps; ++r) {
        GTN_CHECK_HIP(hipEventRecord(e0, s));
        int rc = gemm_grouped_impl(groups, n, dtype, prec, s, nullptr, 0, "gtn_gemm_grouped", tile, target, nullptr, tri, pipe);
        if (rc) return rc;
        GTN_CHECK_HIP(hipEventRecord(e1, s));
        GTN_CHECK_HIP(hipEventSynchronize(e1));
        float ms = 0;
        GTN_CHECK_HIP(hipEventElapsedTime(&ms, e0, e1));
        if (ms < *best) *best = ms;
    }
    return GTN_OK;
}

// the tuned configuration of this signature, if any (no timing)
static int tuned_lookup(const gtn_gemm_desc *groups, int n, int dtype, int prec, int *tile, int *target, int *pipe, bool *found,
                        int kind = kPlain) {
    *tile = 0;
    *target = -1;
    *pipe = kind == kIndirect ? 0 : -1;
    *found = false;
    if (!autotune_on() || dry_run() || n <= 0) return GTN_OK;
    int dev;
    GTN_CHECK_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> l(g_tune_mu);
    auto it = g_tuned.find(tune_key(groups, n, dtype, prec, dev, kind));
    if (it != g_tuned.end()) {
        *tile = it->second.tile;
        *target = it->second.target;
        *pipe = it->second.pipe;
        *found = true;
    }
    return GTN_OK;
}

static int tuned_config(const gtn_gemm_desc *groups, int n, int dtype, int prec, hipStream_t s, int *tile, int *target,
                        int *pipe, int kind = kPlain) {
    const bool tri = kind == kTri;
    bool found;
    int rc0 = tuned_lookup(groups, n, dtype, prec, tile, target, pipe, &found, kind);
    if (rc0 || found || !autotune_on() || dry_run() || n <= 0) return rc0;
    int dev;
    GTN_CHECK_HIP(hipGetDevice(&dev));
    const std::string key = tune_key(groups, n, dtype, prec, dev, kind);
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    GTN_CHECK_HIP(hipStreamIsCapturing(s, &cs));
    if (cs != hipStreamCaptureStatusNone || capture_open()) return GTN_OK;
    bool can128 = true;
    for (int i = 0; i < n; ++i) {
        if (groups[i].beta != 0.0) return GTN_OK;
        if (groups[i].M == 0 || groups[i].N == 0 || groups[i].batch == 0) continue;
        if (groups[i].M < 128 || groups[i].N < 128) can128 = false;
    }
    hipEvent_t e0, e1;
    GTN_CHECK_HIP(hipEventCreate(&e0));
    GTN_CHECK_HIP(hipEventCreate(&e1));
    TuneCfg best{0, -1, 1e30f, 0, 0};
    float ms_default = 0;
    int rc = time_cfg(groups, n, dtype, prec, s, 0, -1, e0, e1, &ms_default, tri, kind == kIndirect ? 0 : -1);
    const int tiles[2] = {64, 128};
    const int targets[4] = {0, 512, 1024, 2048};
    for (int ti = 0; ti < 2 && !rc; ++ti) {
        if (tiles[ti] == 128 && !can128) continue;
        for (int gi = 0; gi < 4 && !rc; ++gi) {
            float ms;
            rc = time_cfg(groups, n, dtype, prec, s, tiles[ti], targets[gi], e0, e1, &ms, tri, 0);
            if (!rc && ms < best.ms) best = TuneCfg{tiles[ti], targets[gi], ms, 0, 0};
        }
    }
    if ((prec == GTN_PREC_F64 && kind != kIndirect) || (prec == GTN_PREC_F32 && dtype == GTN_F32)) {
        const int tried[2] = {best.target, split_target()};
        for (int t = 0; t < (tried[0] == tried[1] ? 1 : 2); ++t)
            for (int ti = 0; ti < 2 && !rc; ++ti) {
                if (tiles[ti] == 128 && !can128) continue;
                float ms;
                rc = time_cfg(groups, n, dtype, prec, s, tiles[ti], tried[t], e0, e1, &ms, tri, 1);
                if (!rc && ms < best.ms) best = TuneCfg{tiles[ti], tried[t], ms, 0, 1};
            }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    best.ms_default = ms_default;
    std::lock_guard<std::mutex> l(g_tune_mu);
    g_tuned[key] = best;
    *tile = best.tile;
    *target = best.target;
    *pipe = best.pipe;
    return GTN_OK;
}

extern "C" int gtn_gemm_grouped(const gtn_gemm_desc *groups, int n_groups, int dtype, int precision, void *stream) {
    int tile = 0, target = -1, pipe = -1;
    int rc = tuned_config(groups, n_groups, dtype, precision, as_stream(stream), &tile, &target, &pipe);
    if (rc) return rc;
    return gemm_grouped_impl(groups, n_groups, dtype, precision, stream, nullptr, 0, "gtn_gemm_grouped", tile, target,
                             nullptr, false, pipe);
}

extern "C" int gtn_gemm_grouped_as(const gtn_gemm_desc *groups, int n_groups, int dtype, int precision, int tile,
                                   int split_target, int kernel, int symmetric, void *stream) {
    GTN_REQUIRE(n_groups >= 0 && (n_groups == 0 || groups), "gtn_gemm_grouped_as: bad groups");
    GTN_REQUIRE((tile == 64 || tile == 128) && split_target >= 0 && split_target <= 4096 && (kernel == 0 || kernel == 1),
                "gtn_gemm_grouped_as: bad configuration");
    GTN_REQUIRE(kernel == 0 || precision == GTN_PREC_F64 || (precision == GTN_PREC_F32 && dtype == GTN_F32),
                "gtn_gemm_grouped_as: this precision has one kernel");
    GTN_REQUIRE(!symmetric || (dtype == GTN_F64 && precision == GTN_PREC_F64), "gtn_gemm_grouped_as: symmetric products are FP64");
    for (int i = 0; i < n_groups; ++i) {
        const gtn_gemm_desc &d = groups[i];
        if (d.M == 0 || d.N == 0 || d.batch == 0) continue;
        GTN_REQUIRE(tile == 64 || (d.M >= 128 && d.N >= 128), "gtn_gemm_grouped_as: a group below the tile's size");
        GTN_REQUIRE(!symmetric || (d.M == d.N && d.beta == 0.0), "gtn_gemm_grouped_as: not a symmetric product");
    }
    return gemm_grouped_impl(groups, n_groups, dtype, precision, stream, nullptr, 0, "gtn_gemm_grouped_as", tile, split_target,
                             nullptr, symmetric != 0, kernel);
}

int gtn::gemm_symmetric(const gtn_gemm_desc *groups, int n_groups, void *stream) {
    for (int i = 0; i < n_groups; ++i)
        GTN_REQUIRE(groups[i].M == groups[i].N, "gtn_svd_blocks: a symmetric product is square");
    int tile = 0, target = -1, pipe = -1;
    int rc = tuned_config(groups, n_groups, GTN_F64, GTN_PREC_F64, as_stream(stream), &tile, &target, &pipe, kTri);
    if (rc) return rc;
    return gemm_grouped_impl(groups, n_groups, GTN_F64, GTN_PREC_F64, stream, nullptr, 0, "gtn_svd_blocks", tile, target,
                             nullptr, true, pipe);
}

int gtn::gemm_grouped_indirect(const gtn_gemm_desc *groups, const GemmIndirect *ind, int n_groups, void *const *tune_c,
                               void *stream) {
    int tile = 0, target = -1, pipe = 0, rc;
    if (tune_c) {
        std::vector<gtn_gemm_desc> plain(groups, groups + n_groups);
        for (int i = 0; i < n_groups; ++i) plain[i].C = tune_c[i];
        rc = tuned_config(plain.data(), n_groups, GTN_F64, GTN_PREC_F64, as_stream(stream), &tile, &target, &pipe, kIndirect);
    } else {
        bool found;
        rc = tuned_lookup(groups, n_groups, GTN_F64, GTN_PREC_F64, &tile, &target, &pipe, &found, kIndirect);
    }
    if (rc) return rc;
    return gemm_grouped_impl(groups, n_groups, GTN_F64, GTN_PREC_F64, stream, nullptr, 0, "gtn_svd_blocks", tile, target, ind, false, 0);
}

extern "C" int gtn_autotune_set(int on) {
    g_autotune = on ? 1 : 0;
    return GTN_OK;
}

extern "C" int gtn_autotune_clear(void) {
    std::lock_guard<std::mutex> l(g_tune_mu);
    g_tuned.clear();
    return GTN_OK;
}

extern "C" int gtn_autotune_report(gtn_tune_entry *out, int max_entries) {
    std::lock_guard<std::mutex> l(g_tune_mu);
    int i = 0;
    for (auto &kv : g_tuned) {
        if (!out || i >= max_entries) break;
        const int64_t *k = (const int64_t *)kv.first.data();
        gtn_tune_entry &e = out[i++];
        memset(&e, 0, sizeof(e));
        e.dtype = (int32_t)k[1];
        e.precision = (int32_t)k[2];
        e.n_groups = (int32_t)k[3];
        e.M = k[4];
        e.N = k[5];
        e.K = k[6];
        e.batch = k[7];
        e.tile = kv.second.tile;
        e.split_target = kv.second.target;
        e.kernel = kv.second.pipe;
        e.ms_best = kv.second.ms;
        e.ms_default = kv.second.ms_default;
    }
    return (int)g_tuned.size();
}

extern "C" int64_t gtn_gemm_noalloc_max_scratch(void) { return kNoAllocScratchBytes; }

// Follows gtn_gemm_grouped's tuned configuration of the signature (never timing one itself), unless
// that configuration's split plan would not fit the scratch: then the heuristics, whose split plans
// always fit (at most ~2 x 1024 workgroups of 64 x 64 FP64 partials = 64 MiB).
extern "C" int gtn_gemm_grouped_noalloc(const gtn_gemm_desc *groups, int n_groups, int dtype, int precision,
                                        void *stream) {
    void *p = nullptr;
    int rc = scratch_ptr(&p);
    if (rc) return rc;
    int tile = 0, target = -1, pipe = -1;
    bool found = false;
    rc = tuned_lookup(groups, n_groups, dtype, precision, &tile, &target, &pipe, &found);
    if (rc) return rc;
    if (found && target > 1024) {
        // a larger split target than the heuristics' may need more scratch than there is
        rc = gemm_grouped_impl(groups, n_groups, dtype, precision, stream, p, kNoAllocScratchBytes,
                               "gtn_gemm_grouped_noalloc", tile, target, nullptr, false, pipe);
        if (rc != GTN_ENOMEM) return rc;
        tile = 0;
        target = pipe = -1;
    }
    return gemm_grouped_impl(groups, n_groups, dtype, precision, stream, p, kNoAllocScratchBytes,
                             "gtn_gemm_grouped_noalloc", tile, target, nullptr, false, pipe);
}

// int8 16x16x64 lane-layout self-test (the operands are deterministic small integers; one wavefront)
typedef int i32x4 __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(64) k_mfma_selftest_i8(int32_t *out) {
    const int l = threadIdx.x;
    if (l >= 64) return;
    int8_t av[16], bv[16];
    for (int t = 0; t < 16; ++t) {
        const int k = 16 * (l / 16) + t;
        av[t] = (int8_t)(((l % 16) + 3 * k) % 7 - 3);
        bv[t] = (int8_t)((2 * (l % 16) + k) % 5 - 2);
    }
    i32x4 a, b;
    memcpy(&a, av, 16);
    memcpy(&b, bv, 16);
    i32x4 acc = {0, 0, 0, 0};
    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, acc, 0, 0, 0);
    for (int v = 0; v < 4; ++v) out[4 * l + v] = acc[v];
}

extern "C" int gtn_mfma_selftest_i8(int32_t *out_dev, void *stream) {
    GTN_REQUIRE(out_dev, "gtn_mfma_selftest_i8: null output");
    hipLaunchKernelGGL(k_mfma_selftest_i8, dim3(1), dim3(64), 0, as_stream(stream), out_dev);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

extern "C" int gtn_mfma_selftest(double *out_dev, void *stream) {
    GTN_REQUIRE(out_dev, "gtn_mfma_selftest: null output");
    hipLaunchKernelGGL(k_mfma_selftest, dim3(1), dim3(64), 0, as_stream(stream), out_dev);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}
