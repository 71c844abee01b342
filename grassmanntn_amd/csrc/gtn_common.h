// Internal helpers shared by the HIP translation units of libgtn_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include "../../include/gtn_hip.h"

namespace gtn {

// Thread-local message behind gtn_last_error().
void set_error(const char *fmt, ...);

#define GTN_CHECK_HIP(expr)                                                              \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess) {                                                          \
            gtn::set_error("%s:%d %s: %s", __FILE__, __LINE__, #expr, hipGetErrorString(e_)); \
            return GTN_EDEVICE;                                                          \
        }                                                                                \
    } while (0)

#define GTN_REQUIRE(cond, ...)            \
    do {                                  \
        if (!(cond)) {                    \
            gtn::set_error(__VA_ARGS__);  \
            return GTN_EINVAL;            \
        }                                 \
    } while (0)

// Launch-error check after a kernel launch.
#define GTN_CHECK_LAUNCH() GTN_CHECK_HIP(hipGetLastError())

__device__ __forceinline__ uint32_t popc64(uint64_t x) { return (uint32_t)__popcll(x); }
// eps(i) = i ^ (popcount(i >> 1) & 1): canonical <-> parity-preserving (an involution)
__device__ __forceinline__ uint64_t enc_switch(uint64_t i) { return i ^ (uint64_t)(popc64(i >> 1) & 1u); }
// sigma(i) = -1 iff popcount(i) mod 4 is 2 or 3; returned as a sign bit (1 => negative)
__device__ __forceinline__ uint32_t sigma_bit(uint64_t i) { return (popc64(i) >> 1) & 1u; }

// dry-run validation (host only): registered regions and a range check
bool dry_run();
int check_range(const void *p, int64_t bytes, const char *what);
#define GTN_RANGE(p, bytes, what)                         \
    do {                                                  \
        int rc_ = gtn::check_range((p), (bytes), (what)); \
        if (rc_) return rc_;                              \
    } while (0)

// Operands and epilogue of a grouped FP64 GEMM whose batch entries keep them on the device (the range
// finder of gtn_svd_blocks, whose blocks stop and trade buffers one by one).  Per batch entry, `stride`
// 8-byte slots apart: the operand pointers (a null table: the descriptor's pointer and batch stride) and
// coef = {x, y, z, skip}: C = x A B + y D + z C, D of C's shape and strides; nothing happens when
// skip is nonzero.
struct GemmIndirect {
    const double *const *a, *const *b, *const *d;
    double *const *c;
    const double *coef;
    int64_t stride;
};
// gtn_gemm_grouped over such groups (alpha and beta of the descriptors are not used); the launch
// configuration is the one tuned for the plain signature, tried out with `tune_c` (same shape, free to
// be overwritten) as output; tune_c null: nothing is tried out
int gemm_grouped_indirect(const gtn_gemm_desc *groups, const GemmIndirect *ind, int n_groups, void *const *tune_c,
                          void *stream);

// gtn_gemm_grouped over FP64 products A B that are symmetric (B = A^T; M = N, beta = 0): only the tiles on
// and above the diagonal are computed, (1 + 1 / tiles) / 2 of the product, and stored on both sides
int gemm_symmetric(const gtn_gemm_desc *groups, int n_groups, void *stream);

// While one of these lives, the event that orders other streams behind this thread's split reductions is
// recorded once, by finish() (or the destructor), or by whoever uses their workspace on another stream before
// that: a record between two launches leaves the device idle for 5.6 us, and a decomposition has
// 50 split reductions.  The streams used live at least as long.  No lock is held between the reductions.
class SplitScope {
public:
    SplitScope();
    ~SplitScope() { (void)finish(); }
    int finish();
    SplitScope(const SplitScope &) = delete;
    SplitScope &operator=(const SplitScope &) = delete;

private:
    bool outer_;  // an enclosing scope of this thread does the work
    bool open_ = true;
};

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

// graph bookkeeping of the runtime (gtn_runtime.hip): instantiated graphs that may still be
// launched, and whether a capture is open.  Library-owned device buffers that a graph may hold are
// never freed or moved while either is nonzero.
int graphs_alive();
int capture_open();

inline int grid_for(int64_t n, int block, int max_blocks = 65536) {
    int64_t g = (n + block - 1) / block;
    if (g > max_blocks) g = max_blocks;
    if (g < 1) g = 1;
    return (int)g;
}

}  // namespace gtn
