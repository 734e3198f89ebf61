// kq_sample.hip — greedy sampling on device: the index of the largest logit.
//
// Rule of the engine's greedy sampler (vendor/katali_gguf_dense/src/
// gguf_sampler.c:62-66): best = 0, bv = -FLT_MAX, then for i ascending take i
// when logits[i] > bv. So the first maximum wins, NaN never wins, and when no
// value exceeds -FLT_MAX the answer is 0. Here: (value, index) pairs reduced
// with "larger value, then lower index" over candidates v > -FLT_MAX, in one
// launch: every workgroup reduces its share and stores its pair as one
// device-coherent 64-bit word; once that store is acknowledged it counts
// itself in, and the workgroup that counts last reduces the partials and
// writes the answer, then puts the count back to zero for the next call
// (stream order: no two calls overlap, and a graph replay starts from zero).
#include <float.h>

#include "kq_device.h"
#include "kq_launch.h"

namespace kq {

constexpr int32_t NONE = 0x7FFFFFFF;

struct Best {
    float v;
    int32_t i;
};
__device__ __forceinline__ Best better(Best a, Best b) {
    return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}
// On the VALU (DPP, permlane swaps): the wave's largest value, then the
// lowest index that holds it. Values are never NaN; -0 and +0 compare equal.
__device__ __forceinline__ Best wave_best(Best b) {
    float m = b.v;
    m = fmaxf(m, dpp_f<DPP_XOR1>(m));
    m = fmaxf(m, dpp_f<DPP_XOR2>(m));
    m = fmaxf(m, dpp_f<DPP_HALF_MIRROR>(m));
    m = fmaxf(m, dpp_f<DPP_MIRROR>(m));
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    m = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    m = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    int i = b.v == m ? b.i : NONE;
    i = min(i, dpp_i<DPP_XOR1>(i));
    i = min(i, dpp_i<DPP_XOR2>(i));
    i = min(i, dpp_i<DPP_HALF_MIRROR>(i));
    i = min(i, dpp_i<DPP_MIRROR>(i));
    r = __builtin_amdgcn_permlane16_swap((uint32_t)i, (uint32_t)i, false, false);
    i = min((int)r[0], (int)r[1]);
    r = __builtin_amdgcn_permlane32_swap((uint32_t)i, (uint32_t)i, false, false);
    i = min((int)r[0], (int)r[1]);
    return Best{m, i};
}
__device__ __forceinline__ Best block_best(Best b) {
    __shared__ Best part[4];
    b = wave_best(b);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = b;
    __syncthreads();
    b = part[0];
#pragma unroll
    for (int w = 1; w < 4; w++) b = better(b, part[w]);
    return b;
}

constexpr uint32_t ARGMAX_PARTS = 256;
constexpr uint32_t ARGMAX_COUNT = 2 * ARGMAX_PARTS;   // the count word, after the partials

__device__ __forceinline__ uint64_t pack(Best b) { return ((uint64_t)(uint32_t)b.i << 32) | __float_as_uint(b.v); }
__device__ __forceinline__ Best unpack(uint64_t w) { return Best{__uint_as_float((uint32_t)w), (int32_t)(w >> 32)}; }

// words: ARGMAX_PARTS 64-bit partials, then the count (zero between calls)
template <uint32_t ARGMAX_U>
__global__ void __launch_bounds__(256) k_argmax(const float *__restrict__ x, uint32_t n, uint32_t *words,
                                                int32_t *out) {
    __shared__ uint32_t last;
    Best b{-FLT_MAX, NONE};
    // ascending t per thread: strict > keeps the first. ARGMAX_U loads in flight
    // per round (positions past n load x[n - 1] and are dropped).
    for (uint32_t t0 = blockIdx.x * 256 + threadIdx.x, st = gridDim.x * 256; t0 < n;) {
        float v[ARGMAX_U];
        const uint32_t left = (n - 1 - t0) / st;   // positions t0 + st k, k <= left, are in range
#pragma unroll
        for (uint32_t k = 0; k < ARGMAX_U; k++) v[k] = x[k <= left ? t0 + st * k : n - 1];
#pragma unroll
        for (uint32_t k = 0; k < ARGMAX_U; k++)
            if (k <= left && v[k] > b.v) b = Best{v[k], (int32_t)(t0 + st * k)};
        if (left < ARGMAX_U) break;
        t0 += st * ARGMAX_U;
    }
    b = block_best(b);
    if (threadIdx.x == 0) {
        st_dev2(words + 2 * blockIdx.x, pack(b));
        __builtin_amdgcn_s_waitcnt(VMCNT0);   // the partial is acknowledged before the count
        last = __hip_atomic_fetch_add(words + ARGMAX_COUNT, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
               gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    Best r{-FLT_MAX, NONE};
    for (uint32_t t = threadIdx.x; t < gridDim.x; t += 256) r = better(r, unpack(ld_dev2(words + 2 * t)));
    r = block_best(r);
    if (threadIdx.x == 0) {
        *out = r.i == NONE ? 0 : r.i;
        st_dev(words + ARGMAX_COUNT, 0u);
    }
}

uint32_t argmax_scratch_bytes() { return 4 * (ARGMAX_COUNT + 1); }

hipError_t launch_argmax(const float *x, uint32_t n, void *scratch, int32_t *out, hipStream_t s) {
    auto go = [&](auto kern, uint32_t per) -> hipError_t {   // one round of `per` elements per workgroup, if it can
        uint32_t g = (n + per - 1) / per;
        if (g < 1) g = 1;
        if (g > ARGMAX_PARTS) g = ARGMAX_PARTS;
        hipLaunchKernelGGL(kern, dim3(g), dim3(256), 0, s, x, n, (uint32_t *)scratch, out);
        return hipGetLastError();
    };
    // Half as many workgroups of eight loads a thread where they are many: each
    // costs the count word an atomic and the last one a partial (65536: 3.76 us,
    // with four loads 3.89; 151936: 4.14 and 4.84; 256000: 4.73 and 6.03).
    return n < 65536 ? go(k_argmax<4>, 1024) : go(k_argmax<8>, 2048);
}

}  // namespace kq
