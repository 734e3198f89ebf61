// kq_norm.hip — the decode chain's RMSNorm and residual add on device.
//
// Arithmetic of the engine (vendor/katali_gguf_dense/src/gguf_kernels.c:13-18):
// sumsq = sum of x[i]^2 in double, inv = 1 / sqrtf((float)(sumsq / n) + eps),
// out[i] = x[i] * inv * w[i] (two float products, no contraction). The
// residual step before a norm (gguf_model.c:677-678, 692-693) is x[i] +=
// delta[i], or x[i] += scale * delta[i] when the model scales its residual.
//
// One workgroup of 1024 threads: each thread adds and squares its elements
// (t, t + 1024, ...), the double partial sums meet in a fixed tree (a DPP
// and permlane butterfly in each wave, then the 16 wave sums in order), every
// thread forms the same inv and writes its outputs. The double sum is in a different order than the
// engine's loop; its rounding to float is the same unless the two doubles
// straddle a float rounding boundary (relative distance ~2^-29).
//
// Latency-bound: a launch, one load round trip, the tree, one store. Up to
// 8192 elements a thread's x, delta and w are all in flight at once and stay
// in registers (K elements per thread); a loop made each element's loads wait
// for the store of the one before it (x and delta may be one buffer, so the
// compiler cannot reorder them), a memory round trip each.
#include "kq_device.h"
#include "kq_launch.h"

namespace kq {

constexpr uint32_t NORM_THREADS = 1024;

// K > 0: n <= 1024 K, the elements held in registers; K = 0: any n, in a loop
template <bool ADD, int K>
__global__ void __launch_bounds__(NORM_THREADS)
    k_rmsnorm(float *x, const float *delta, float scale, uint32_t unit_scale,
              const float *w, uint32_t n, float eps, float *out) {
    __shared__ double part[NORM_THREADS / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double s = 0.0;
    float v[K > 0 ? K : 1], dv[K > 0 ? K : 1], wv[K > 0 ? K : 1];
    if constexpr (K > 0) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint32_t i = min(tid + NORM_THREADS * k, n - 1);   // clamped, not skipped
            v[k] = x[i];
            if constexpr (ADD) dv[k] = delta[i];
        }
#pragma unroll
        for (int k = 0; k < K; k++) wv[k] = w[min(tid + NORM_THREADS * k, n - 1)];
        // every load is out before the first store (which a buffer it loads
        // from may share, element by element); the sums wait for x and delta only
        asm volatile("" ::: "memory");
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint32_t i = tid + NORM_THREADS * k;
            if constexpr (ADD) {
                v[k] = unit_scale ? v[k] + dv[k] : v[k] + scale * dv[k];
                if (i < n) x[i] = v[k];
            }
            if (i < n) s += (double)v[k] * (double)v[k];
        }
    } else {
        for (uint32_t i = tid; i < n; i += NORM_THREADS) {
            float e = x[i];
            if constexpr (ADD) {
                e = unit_scale ? e + delta[i] : e + scale * delta[i];
                x[i] = e;
            }
            s += (double)e * (double)e;
        }
    }
    s = wave_sum_f64(s);
    if (lane == 0) part[wave] = s;
    __syncthreads();
    double sumsq = part[0];
#pragma unroll
    for (uint32_t k = 1; k < NORM_THREADS / 64; k++) sumsq += part[k];
    const float inv = 1.0f / sqrtf((float)(sumsq / (double)n) + eps);
    if constexpr (K > 0) {
#pragma unroll
        for (int k = 0; k < K; k++)
            if (tid + NORM_THREADS * k < n) out[tid + NORM_THREADS * k] = v[k] * inv * wv[k];
    } else {
        for (uint32_t i = tid; i < n; i += NORM_THREADS) out[i] = x[i] * inv * w[i];   // this thread's own x[i]
    }
}

template <bool ADD>
static hipError_t norm_run(float *x, const float *delta, float scale, const float *w, uint32_t n, float eps, float *out,
                           hipStream_t s) {
    const uint32_t unit = scale == 1.0f ? 1u : 0u;
    auto go = [&](auto kern) -> hipError_t {
        hipLaunchKernelGGL(kern, dim3(1), dim3(NORM_THREADS), 0, s, x, delta, scale, unit, w, n, eps, out);
        return hipGetLastError();
    };
    // a weight vector that the residual step updates is read behind the update
    if (ADD && w < x + n && x < w + n) return go(k_rmsnorm<ADD, 0>);
    if (n <= NORM_THREADS) return go(k_rmsnorm<ADD, 1>);
    if (n <= 2 * NORM_THREADS) return go(k_rmsnorm<ADD, 2>);
    if (n <= 4 * NORM_THREADS) return go(k_rmsnorm<ADD, 4>);
    if (n <= 8 * NORM_THREADS) return go(k_rmsnorm<ADD, 8>);
    return go(k_rmsnorm<ADD, 0>);
}

hipError_t launch_rmsnorm(const float *x, const float *w, uint32_t n, float eps, float *out, hipStream_t s) {
    return norm_run<false>((float *)x, nullptr, 1.0f, w, n, eps, out, s);
}

hipError_t launch_add_rmsnorm(float *x, const float *delta, float scale, const float *w, uint32_t n, float eps,
                              float *out, hipStream_t s) {
    return norm_run<true>(x, delta, scale, w, n, eps, out, s);
}

}  // namespace kq
