// kq_items.h — lane items against an activation staged in item order, and the
// launch helpers of the kernels built on them (the dense GEMV and the wide
// down projection).
#pragma once

#include <type_traits>

#include "kq_device.h"
#include "kq_launch.h"

namespace kq {

// An activation in LDS, laid out for the lanes that read it. A lane item takes
// NQ groups of 16 values (Q4_K: sub-blocks 2g and 2g+1; Q6_K: quarters t = 0..3
// of a half). Tiles of 16 items hold word after word
// of each group side by side for the 16 items, so the lanes of a row read
// consecutive 16-byte words at offsets the instruction carries; in the
// activation's own order they are 64 (fp32) or up to 128 (q8_1) bytes apart,
// a 4-way bank conflict on every read.
//   MODE 0     float4 [4 NQ words][16 items], then the groups' sums (left to
//              right) float [NQ][16]; words 288 bytes apart, so that the eight
//              lanes storing one 32-value run hit distinct banks
//   MODE 1, 2  int8 x 16 [NQ][16], the q8_1 blocks' d float [NQ][8], the
//              groups' exact sums int [NQ][16]: 352 bytes per 256 values, as
//              in the activation's own order
template <class QT, int MODE>
struct XLds {
    static constexpr uint32_t NQ = 16 / QT::IPB;
    static constexpr uint32_t WORD = MODE == 0 ? 288 : 256;
    static constexpr uint32_t D8 = NQ * WORD, SUM = MODE == 0 ? 4 * NQ * WORD : D8 + NQ * 32;
    static constexpr uint32_t TILE = SUM + NQ * 64;
    static constexpr uint32_t bytes(uint32_t items) { return (items + 15) / 16 * TILE; }
    // the item and group of 16-value run h (counted along the activation)
    __device__ static __forceinline__ void place(uint32_t h, uint32_t &item, uint32_t &q) {
        if constexpr (QT::TYPE == T_Q4_K) {   // h = 16 b + 4 g + 2 q + hh
            q = (h >> 1) & 1;
            item = ((h >> 2) << 1) | (h & 1);
        } else {                              // h = 16 b + 8 n + 2 q + k
            q = (h >> 1) & 3;
            item = ((h >> 3) << 1) | (h & 1);
        }
    }
    uint8_t *t;   // the item's tile
    uint32_t l;   // the item in it
    __device__ __forceinline__ XLds(uint8_t *lds, uint32_t item) : t(lds + (item >> 4) * TILE), l(item & 15) {}
    __device__ __forceinline__ float4 *xf(uint32_t word) const { return (float4 *)(t + word * WORD + l * 16); }
    __device__ __forceinline__ float *fsum(uint32_t q) const { return (float *)(t + SUM + q * 64 + l * 4); }
    __device__ __forceinline__ int4 *xq(uint32_t q) const { return (int4 *)(t + q * WORD + l * 16); }
    __device__ __forceinline__ float *d8(uint32_t q) const { return (float *)(t + D8 + q * 32 + (l >> 1) * 4); }
    __device__ __forceinline__ int *isum(uint32_t q) const { return (int *)(t + SUM + q * 64 + l * 4); }
};

// fp32 contribution of one lane item (chunk c of a block) against the staged
// activation: the block formats' own arithmetic (Q4K, Q6K in kq_device.h),
// the activation read through XLds.
template <int MODE>
__device__ __forceinline__ float item_dot(const Q4K::Raw &r, int c, const XLds<Q4K, MODE> &x) {
    const int g = c >> 1;
    float ds0, ds1, dm0, dm1;
    Q4K::scales(r, g, ds0, ds1, dm0, dm1);
    if constexpr (MODE == 0) {
        const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        float al = 0.0f, ah = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float4 vl = *x.xf(j), vh = *x.xf(4 + j);
            const uint32_t lo = q[j] & 0x0F0F0F0Fu, hi = (q[j] >> 4) & 0x0F0F0F0Fu;
            al = fmaf((float)(lo & 0xFFu), vl.x, al);
            al = fmaf((float)((lo >> 8) & 0xFFu), vl.y, al);
            al = fmaf((float)((lo >> 16) & 0xFFu), vl.z, al);
            al = fmaf((float)(lo >> 24), vl.w, al);
            ah = fmaf((float)(hi & 0xFFu), vh.x, ah);
            ah = fmaf((float)((hi >> 8) & 0xFFu), vh.y, ah);
            ah = fmaf((float)((hi >> 16) & 0xFFu), vh.z, ah);
            ah = fmaf((float)(hi >> 24), vh.w, ah);
        }
        return fmaf(ds0, al, -(dm0 * *x.fsum(0))) + fmaf(ds1, ah, -(dm1 * *x.fsum(1)));
    } else {
        int slo, shi;
        Q4K::isums_x(r.q, *x.xq(0), *x.xq(1), slo, shi);
        const float vlo = fmaf(ds0, (float)slo, -(dm0 * (float)*x.isum(0)));
        const float vhi = fmaf(ds1, (float)shi, -(dm1 * (float)*x.isum(1)));
        return fmaf(*x.d8(0), vlo, *x.d8(1) * vhi);
    }
}
template <int MODE>
__device__ __forceinline__ float item_dot(const Q6K::Raw &r, int c, const XLds<Q6K, MODE> &x) {
    const int k = c & 1;
    const uint32_t A[4] = {r.A.x, r.A.y, r.A.z, r.A.w};
    const uint32_t B[4] = {r.B.x, r.B.y, r.B.z, r.B.w};
    const uint32_t H[4] = {r.H.x, r.H.y, r.H.z, r.H.w};
    const float d = h2f(r.d);
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        if constexpr (MODE == 0) {
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t v = Q6K::q6(A[j], B[j], H[j], t);
                const float4 w = *x.xf(4 * t + j);
                s = fmaf((float)(v & 0xFFu), w.x, s);
                s = fmaf((float)((v >> 8) & 0xFFu), w.y, s);
                s = fmaf((float)((v >> 16) & 0xFFu), w.z, s);
                s = fmaf((float)(v >> 24), w.w, s);
            }
            s = fmaf(-32.0f, *x.fsum(t), s);
            acc = fmaf(d * Q6K::scale(r, k, t), s, acc);
        } else {
            const int4 w = *x.xq(t);
            int s = dot4(Q6K::q6(A[0], B[0], H[0], t), w.x, 0);
            s = dot4(Q6K::q6(A[1], B[1], H[1], t), w.y, s);
            s = dot4(Q6K::q6(A[2], B[2], H[2], t), w.z, s);
            s = dot4(Q6K::q6(A[3], B[3], H[3], t), w.w, s);
            s -= 32 * *x.isum(t);
            const float v = (d * Q6K::scale(r, k, t)) * (float)s;
            acc = t == 0 ? *x.d8(t) * v : fmaf(*x.d8(t), v, acc);
        }
    }
    return acc;
}

// An entry of the batched layer: up to GRP_MAX (token, rank) pairs of one
// expert, listed as a record of GRP_REC ints.
constexpr uint32_t GRP_MAX = 8;
struct GrpEntry {
    uint32_t ex, cnt;   // uniform
    uint32_t pair;      // lane l: pair l % GRP_MAX (pair 0 past the count)
};
// The record of entry ei; cnt 0 when the list has no such entry (the record is
// inside the list's memory all the same).
__device__ __forceinline__ GrpEntry grp_entry(const MoeArgs &a, uint32_t ei) {
    const int32_t *rec = a.bslot + (uint64_t)GRP_REC * ei;
    const int32_t n = *a.bcount, ex = rec[0], cnt = rec[1];
    GrpEntry e;
    e.pair = (uint32_t)rec[4 + (threadIdx.x & (GRP_MAX - 1))];
    e.ex = (uint32_t)__builtin_amdgcn_readfirstlane(ex);
    e.cnt = ei < (uint32_t)__builtin_amdgcn_readfirstlane(n) ? (uint32_t)__builtin_amdgcn_readfirstlane(cnt) : 0u;
    return e;
}

inline int ilog2(uint32_t v) {
    int l = 0;
    while ((1u << (l + 1)) <= v) l++;
    return l;
}

// f(integral_constant<int, N>) for the run-time N in 1..MAX
template <int MAX, class F>
inline hipError_t with_n(uint32_t n, F &&f) {
    if constexpr (MAX > 1)
        if (n < (uint32_t)MAX) return with_n<MAX - 1>(n, f);
    return f(std::integral_constant<int, MAX>{});
}

template <class Kern>
inline hipError_t lds_limit(Kern kern, uint32_t lds) {
    if (lds <= 64 * 1024) return hipSuccess;
    return hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

}  // namespace kq
