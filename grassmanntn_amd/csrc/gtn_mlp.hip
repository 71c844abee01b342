// Elementwise stages of an ensemble of MLPs (the learned surrogate of the coupling sweep; no
// counterpart in the reference).  The matrix products run on the grouped GEMM of gtn_gemm.hip in
// its BF16 modes; the kernels here are the rest of a training or inference step: bias + GELU with
// the pre-activation kept for the backward pass, the GELU derivative, bias gradients, a weighted
// mean-squared error, AdamW with a cosine learning-rate schedule, and the ensemble mean / spread.
//
// Layout: an ensemble of E members holds, per layer, activations as E row-major (n x c) FP32
// matrices, one after the other.  GELU is x * Phi(x) = 0.5 x (1 + erf(x / sqrt 2)).
#include "gtn_common.h"
#include <math.h>

namespace gtn {

constexpr double kInvSqrt2 = 0.70710678118654752440;
constexpr double kInvSqrt2Pi = 0.39894228040143267794;

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * (float)kInvSqrt2)); }
__device__ __forceinline__ float gelu_grad(float x) {
    return 0.5f * (1.0f + erff(x * (float)kInvSqrt2)) + x * (float)kInvSqrt2Pi * expf(-0.5f * x * x);
}

// The two elementwise passes run over 16-byte vectors where rows and buffers allow it (V = 4; V = 1
// otherwise), without a division an element for the column: at 5 x 4096 x 256 values 14 us became 11
// (bias) and 14 10.5 (derivative), against 10 at the rate of a large copy.
template <int V>
struct alignas(4 * V) Floats {
    float x[V];
};

// y[e][r][j] += bias[e][j]; pre = y (optional); y = act(y), in vectors of V.  grid (blocks, E); the
// position of a lane's vector within its row advances by the grid's stride, taken modulo the row once
template <int V>
__global__ void k_bias_act(float *y, int64_t n, int64_t c, const float *bias, int act, float *pre) {
    const int64_t e = blockIdx.y, total = n * c / V, cv = c / V;
    Floats<V> *ye = (Floats<V> *)y + e * total;
    Floats<V> *pe = pre ? (Floats<V> *)pre + e * total : nullptr;
    const Floats<V> *be = (const Floats<V> *)bias + e * cv;
    const int64_t first = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    const int64_t jstep = step % cv;
    int64_t j = first % cv;
    for (int64_t i = first; i < total; i += step) {
        Floats<V> v = ye[i];
        const Floats<V> bj = be[j];
#pragma unroll
        for (int u = 0; u < V; ++u) v.x[u] += bj.x[u];
        if (pe) pe[i] = v;
        if (act == 1) {
#pragma unroll
            for (int u = 0; u < V; ++u) v.x[u] = gelu(v.x[u]);
        }
        ye[i] = v;
        j += jstep;
        if (j >= cv) j -= cv;
    }
}

template <int V>
__global__ void k_act_backward(float *dy, const float *pre, int64_t count) {
    const int64_t total = count / V;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        Floats<V> d = ((const Floats<V> *)dy)[i];
        const Floats<V> p = ((const Floats<V> *)pre)[i];
#pragma unroll
        for (int u = 0; u < V; ++u) d.x[u] *= gelu_grad(p.x[u]);
        ((Floats<V> *)dy)[i] = d;
    }
}

// out[e][j] = sum_r x[e][r][j] in two passes with a fixed summation order (FP64 accumulation).
// Pass 1, grid (ceil(c / 64), E, kColChunks): rows [q n / R, (q + 1) n / R) of 64 columns; lane ->
// column, the four wavefronts take every fourth row; part[(e R + q) c + j].
constexpr int kColChunks = 32;
__global__ void __launch_bounds__(256) k_colsum_partial(const float *x, int64_t n, int64_t c, double *part) {
    __shared__ double sh[4][64];
    const int64_t e = blockIdx.y, q = blockIdx.z, j = blockIdx.x * 64 + (threadIdx.x & 63);
    const int w = threadIdx.x >> 6;
    const int64_t r0 = q * n / kColChunks, r1 = (q + 1) * n / kColChunks;
    double acc = 0.0;
    if (j < c) {
        const float *xe = x + e * n * c + j;
#pragma unroll 4
        for (int64_t r = r0 + w; r < r1; r += 4) acc += (double)xe[r * c];
    }
    sh[w][threadIdx.x & 63] = acc;
    __syncthreads();
    if (w == 0 && j < c)
        part[(e * kColChunks + q) * c + j] = sh[0][threadIdx.x] + sh[1][threadIdx.x] + sh[2][threadIdx.x] + sh[3][threadIdx.x];
}
__global__ void k_colsum_final(const double *part, int64_t E, int64_t c, float *out) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= E * c) return;
    const int64_t e = t / c, j = t - e * c;
    double acc = 0.0;
    for (int q = 0; q < kColChunks; ++q) acc += part[(e * kColChunks + q) * c + j];
    out[t] = (float)acc;
}

// dout = 2 w_j (out - target) / n; loss[e] = sum_{r,j} w_j (out - target)^2 / n; the target (n x c) is
// shared by the members.  Of a member's workgroups (grid.y, counted from `first`) number 0 sums its loss (in a
// fixed order, four loads in flight a lane), the others, `writers` of them, write dout.  One workgroup of 256 a member that did both,
// an index division and a round trip to memory an element, took 138 us at 4096 x 17 values; this takes 13.5.
constexpr int kMseBlock = 1024;
__global__ void __launch_bounds__(kMseBlock) k_mse(const float *out, const float *target, const float *w, int64_t n, int64_t c,
                                                   float *dout, double *loss, int first, int writers) {
    __shared__ double sh[kMseBlock / 64];
    const int64_t e = blockIdx.x, total = n * c;
    const float *oe = out + e * total;
    const int number = first + (int)blockIdx.y;
    if (number > 0) {
        float *de = dout + e * total;
        const int64_t step = (int64_t)writers * kMseBlock;
        for (int64_t i = (int64_t)(number - 1) * kMseBlock + threadIdx.x; i < total; i += step) {
            const double d = (double)oe[i] - (double)target[i];
            de[i] = (float)(2.0 * w[i % c] * d / (double)n);
        }
        return;
    }
    if (!loss) return;
    double acc = 0.0;
    const int64_t jstep = kMseBlock % c;
    int64_t j = threadIdx.x % c;
#pragma unroll 4
    for (int64_t i = threadIdx.x; i < total; i += kMseBlock) {
        const double d = (double)oe[i] - (double)target[i];
        acc += w[j] * d * d;
        j += jstep;
        if (j >= c) j -= c;
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) sh[wv] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int i = 0; i < kMseBlock / 64; ++i) t += sh[i];
        loss[e] = t / (double)n;
    }
}

// AdamW (decoupled weight decay) at step t = step[0] + 1 with a cosine learning rate from lr_max
// (t = 1) to lr_min (t = total)
__global__ void k_adamw(float *w, const float *g, float *m, float *v, int64_t count, gtn_adamw_opts o, const double *step) {
    const double t = step[0] + 1.0;
    const double frac = o.total_steps > 1 ? fmin((t - 1.0) / (double)(o.total_steps - 1), 1.0) : 0.0;
    const double lr = o.lr_min + 0.5 * (o.lr_max - o.lr_min) * (1.0 + cos(3.14159265358979323846 * frac));
    const double c1 = 1.0 / (1.0 - pow(o.beta1, t)), c2 = 1.0 / (1.0 - pow(o.beta2, t));
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x) {
        const double gi = g[i];
        const double mi = o.beta1 * m[i] + (1.0 - o.beta1) * gi;
        const double vi = o.beta2 * v[i] + (1.0 - o.beta2) * gi * gi;
        m[i] = (float)mi;
        v[i] = (float)vi;
        const double wi = (double)w[i] * (1.0 - lr * o.weight_decay);
        w[i] = (float)(wi - lr * (mi * c1) / (sqrt(vi * c2) + o.eps));
    }
}

__global__ void k_step_inc(double *step) {
    if (threadIdx.x == 0 && blockIdx.x == 0) step[0] += 1.0;
}

// mean / standard deviation (population, divisor E) over the members of count values each
__global__ void k_ens_stats(const float *out, int64_t E, int64_t count, float *mean, float *sd) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x) {
        double s = 0.0, q = 0.0;
        for (int64_t e = 0; e < E; ++e) s += (double)out[e * count + i];
        const double mu = s / (double)E;
        for (int64_t e = 0; e < E; ++e) {
            const double d = (double)out[e * count + i] - mu;
            q += d * d;
        }
        mean[i] = (float)mu;
        if (sd) sd[i] = (float)sqrt(q / (double)E);
    }
}

}  // namespace gtn

using namespace gtn;

static bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

extern "C" {

int gtn_mlp_bias_act(float *y, int64_t E, int64_t n, int64_t c, const float *bias, int act, float *pre, void *stream) {
    GTN_REQUIRE(E >= 1 && n >= 0 && c >= 1 && y && bias, "gtn_mlp_bias_act: bad argument");
    GTN_REQUIRE(act == GTN_ACT_NONE || act == GTN_ACT_GELU, "gtn_mlp_bias_act: unknown activation %d", act);
    GTN_REQUIRE(E <= 65535, "gtn_mlp_bias_act: too many members");
    if (n == 0) return GTN_OK;
    if (c % 4 == 0 && aligned16(y) && aligned16(bias) && aligned16(pre))
        hipLaunchKernelGGL(k_bias_act<4>, dim3(grid_for(n * c / 4, 256, 4096), (unsigned)E), dim3(256), 0, as_stream(stream), y,
                           n, c, bias, act, pre);
    else
        hipLaunchKernelGGL(k_bias_act<1>, dim3(grid_for(n * c, 256, 4096), (unsigned)E), dim3(256), 0, as_stream(stream), y,
                           n, c, bias, act, pre);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_mlp_act_backward(float *dy, const float *pre, int64_t count, int act, void *stream) {
    GTN_REQUIRE(act == GTN_ACT_GELU, "gtn_mlp_act_backward: only GELU has a derivative pass");
    GTN_REQUIRE(count >= 0 && (count == 0 || (dy && pre)), "gtn_mlp_act_backward: bad argument");
    if (count == 0) return GTN_OK;
    if (count % 4 == 0 && aligned16(dy) && aligned16(pre))
        hipLaunchKernelGGL(k_act_backward<4>, dim3(grid_for(count / 4, 256, 1 << 16)), dim3(256), 0, as_stream(stream), dy, pre,
                           count);
    else
        hipLaunchKernelGGL(k_act_backward<1>, dim3(grid_for(count, 256, 1 << 16)), dim3(256), 0, as_stream(stream), dy, pre,
                           count);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int64_t gtn_mlp_colsum_workspace(int64_t E, int64_t c) { return E * c * kColChunks * (int64_t)sizeof(double); }

int gtn_mlp_colsum(const float *x, int64_t E, int64_t n, int64_t c, float *out, double *part, void *stream) {
    GTN_REQUIRE(E >= 1 && E <= 65535 && n >= 0 && c >= 1 && x && out && part, "gtn_mlp_colsum: bad argument");
    hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(k_colsum_partial, dim3((unsigned)((c + 63) / 64), (unsigned)E, kColChunks), dim3(256), 0, s, x, n,
                       c, part);
    GTN_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_colsum_final, dim3(grid_for(E * c, 256)), dim3(256), 0, s, (const double *)part, E, c, out);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_mlp_mse(const float *out, const float *target, const float *weight, int64_t E, int64_t n, int64_t c, float *dout,
                double *loss, void *stream) {
    GTN_REQUIRE(E >= 1 && n >= 1 && c >= 1 && out && target && weight && dout, "gtn_mlp_mse: bad argument");
    const int writers = grid_for(n * c, kMseBlock, 256);
    hipStream_t s = as_stream(stream);
    auto overlaps = [](const float *a, int64_t na, const float *b, int64_t nb) {
        return (uintptr_t)a < (uintptr_t)(b + nb) && (uintptr_t)b < (uintptr_t)(a + na);
    };
    if (overlaps(dout, E * n * c, out, E * n * c) || overlaps(dout, E * n * c, target, n * c)) {
        // in place: the loss is summed before anything is written
        hipLaunchKernelGGL(k_mse, dim3((unsigned)E, 1), dim3(kMseBlock), 0, s, out, target, weight, n, c, dout, loss, 0, writers);
        GTN_CHECK_LAUNCH();
        hipLaunchKernelGGL(k_mse, dim3((unsigned)E, writers), dim3(kMseBlock), 0, s, out, target, weight, n, c, dout, loss, 1,
                           writers);
    } else {
        hipLaunchKernelGGL(k_mse, dim3((unsigned)E, 1 + writers), dim3(kMseBlock), 0, s, out, target, weight, n, c, dout, loss,
                           0, writers);
    }
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_adamw(float *w, const float *g, float *m, float *v, int64_t count, const gtn_adamw_opts *opts, double *step,
              void *stream) {
    GTN_REQUIRE(count >= 0 && opts && step && (count == 0 || (w && g && m && v)), "gtn_adamw: bad argument");
    GTN_REQUIRE(opts->beta1 >= 0 && opts->beta1 < 1 && opts->beta2 >= 0 && opts->beta2 < 1 && opts->eps > 0,
                "gtn_adamw: bad moments");
    hipStream_t s = as_stream(stream);
    if (count) {
        hipLaunchKernelGGL(k_adamw, dim3(grid_for(count, 256, 4096)), dim3(256), 0, s, w, g, m, v, count, *opts,
                           (const double *)step);
        GTN_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(k_step_inc, dim3(1), dim3(64), 0, s, step);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

int gtn_ensemble_stats(const float *out, int64_t E, int64_t count, float *mean, float *sd, void *stream) {
    GTN_REQUIRE(E >= 1 && count >= 0 && (count == 0 || (out && mean)), "gtn_ensemble_stats: bad argument");
    if (count == 0) return GTN_OK;
    hipLaunchKernelGGL(k_ens_stats, dim3(grid_for(count, 256)), dim3(256), 0, as_stream(stream), out, E, count, mean, sd);
    GTN_CHECK_LAUNCH();
    return GTN_OK;
}

}  // extern "C"
