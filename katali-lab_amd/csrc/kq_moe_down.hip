// kq_moe_down.hip — down projections of long rows: kernel B for rows that none
// of its unrolled variants takes or that fill a wave in several slots, and the
// batched layer's grouped kernel for Q4_K rows above 16 blocks.
//
// Kernel B's: a workgroup takes a run of output rows and all their slots, pair
// (slot, row) after pair with the rows of one slot in a row, so it reads each
// slot's rows as one stretch of memory. A pair is dotted by S lanes of a wave
// (64, or 4 blocks' items for rows of 5 to 16 blocks), N items each per batch
// with all their loads in flight; every slot's h is staged once per workgroup
// in item order (kq_items.h). The partial sums of a pair meet on the VALU, the
// rows' slots in rank order as in kernel B.
//
// Bound by the weight stream; what it had been bound by is the h staging (a
// workgroup of 256 threads staged 32 KB of h for 47 KB of weights at two slots
// of 14336) and, where no unrolled variant fits (Q4_K rows above 16 blocks,
// more than four slots of Q6_K rows above 16), a loop with one block in
// flight per lane.
#include "kq_device.h"
#include "kq_items.h"
#include "kq_launch.h"

namespace kq {

constexpr uint32_t DW_MAX_NT = 1024;
constexpr int DW_HT = 4;            // h tasks per thread in registers ahead of the weights

template <class QD>
constexpr int dw_nmax() { return QD::TYPE == T_Q4_K ? 8 : 4; }
static_assert(XLds<Q4K, 1>::TILE == 16 / Q4K::IPB * 352 && XLds<Q6K, 1>::TILE == 16 / Q6K::IPB * 352,
              "h in item order: the plan's bytes (item_tile_bytes)");

// One 16-byte half block of a slot's h per task: 16 values are one group of
// one item.
struct DwH {
    uint4 q;
    uint32_t d;
};
__device__ __forceinline__ DwH dw_load_h(const uint8_t *hq8, uint32_t t) {
    const uint8_t *b = hq8 + (uint64_t)(t >> 1) * 36;
    DwH h;
    h.q = ld16(b + 4 + 16 * (t & 1));
    h.d = ld_u16(b);
    return h;
}
// run r of the h that starts at item `first`
template <class QD>
__device__ __forceinline__ void dw_put_h(uint8_t *lds, uint32_t first, uint32_t r, const DwH &h) {
    using X = XLds<QD, 1>;
    uint32_t item, grp;
    X::place(r, item, grp);
    const X x(lds, first + item);
    *(uint4 *)x.xq(grp) = h.q;
    int sum = dot4(h.q.x, 0x01010101u, 0);
    sum = dot4(h.q.y, 0x01010101u, sum);
    sum = dot4(h.q.z, 0x01010101u, sum);
    sum = dot4(h.q.w, 0x01010101u, sum);
    *x.isum(grp) = sum;
    if ((r & 1) == 0) *x.d8(grp) = h2f(h.d);   // both halves of a block share it
}

// PACK: the slots' h without gaps (DownPlan). Otherwise a slot starts with a
// tile, and an item's place in it is one for all pairs: formed per pair it cost
// layers of two Q4_K slots 0.1 to 0.2 us of 15 to 17.
template <class QD, int N, bool PACK>
__global__ void __launch_bounds__(DW_MAX_NT) k_moe_down_wide(MoeArgs a, uint32_t rpw, uint32_t inv_rpw, uint32_t n_slots,
                                                              uint32_t log2s) {
    extern __shared__ __align__(16) uint8_t lds[];
    using X = XLds<QD, 1>;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockDim.x;
    const uint32_t nb = a.ffn / 256, items = nb * QD::IPB;
    const uint32_t slot_bytes = PACK ? 0 : X::bytes(items), slot_items = PACK ? items : 0;
    // the normed layer's exchange generation, read now and advanced at the
    // end, as kernel B does
    uint32_t gen = ld_dev(a.router ? a.fsync + 1 : (uint32_t *)a.route_ids);
    const int32_t rid = a.route_ids[min(lane, DW_SLOTS - 1)];
    float rw = a.route_w[min(lane, DW_SLOTS - 1)];
    const uint32_t per = a.ffn / 16, ntask = n_slots * per;
    DwH hv[DW_HT];
#pragma unroll
    for (int i = 0; i < DW_HT; i++) hv[i] = dw_load_h(a.hq8, min(tid + nt * i, ntask - 1));   // clamped, not skipped

    const uint32_t S = 1u << log2s, sp = WAVE >> log2s, s = lane & (S - 1);
    const uint32_t row0 = blockIdx.x * rpw, nrows = min(rpw, a.hidden - row0);
    // pair p: row p % rpw of slot p / rpw (inv_rpw: 2^20 / rpw rounded up);
    // rows past the last one are read as it and dropped at the end
    const uint32_t npairs = rpw * n_slots;
    const uint32_t step = nt / WAVE * sp;   // pairs per round of the workgroup
    const uint64_t rb = (uint64_t)nb * QD::BB;
    uint32_t p = wave * sp + (lane >> log2s);   // this lane-slot's pair; past npairs: the last one, dropped
    typename QD::RawQ raw[N];
    auto load = [&](uint32_t i0) {
        const uint32_t pc = min(p, npairs - 1), sl = pc * inv_rpw >> 20, r = min(pc - sl * rpw, nrows - 1);
        const int32_t sid = __shfl(rid, (int)sl, WAVE);
        const uint8_t *db = (int)sl < a.n_sel ? a.down + (uint64_t)sid * a.hidden * rb : a.down_sh;
        const uint8_t *rp = db + (uint64_t)(row0 + r) * rb;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t item = min(s + S * (i0 + i), items - 1);
            raw[i] = QD::load_quad(rp + (item / QD::IPB) * QD::BB, (int)(item % QD::IPB));
        }
    };
    load(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);   // every weight load is out before h is staged
#pragma unroll
    for (int i = 0; i < DW_HT; i++)
        if (const uint32_t t = tid + nt * i; t < ntask)
            dw_put_h<QD>(lds + t / per * slot_bytes, t / per * slot_items, t % per, hv[i]);
    for (uint32_t t = tid + nt * DW_HT; t < ntask; t += nt)
        dw_put_h<QD>(lds + t / per * slot_bytes, t / per * slot_items, t % per, dw_load_h(a.hq8, t));
    __syncthreads();

    float *res = (float *)(lds + (PACK ? X::bytes(n_slots * items) : n_slots * slot_bytes));   // [row][slot]
    float acc = 0.0f;
    // batches of a pair, then the next pair, in one loop with one load: two
    // loads (or a nested loop) cost a second set of raw registers
    for (uint32_t i0 = 0;;) {
        const uint32_t pc = min(p, npairs - 1), sl = pc * inv_rpw >> 20;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t at = s + S * (i0 + i), item = min(at, items - 1);
            const X x(lds + sl * slot_bytes, sl * slot_items + item);
            const float v = item_dot<1>(QD::full(raw[i]), (int)(item % QD::IPB), x);
            acc += at < items ? v : 0.0f;
            asm volatile("" : "+v"(acc)::"memory");   // one item's h in registers at a time
        }
        i0 += N;
        if (S * i0 >= items) {   // the pair is done
            float v;
            switch (log2s) {   // uniform
                case 6: v = group_sum<64>(acc); break;
                case 5: v = group_sum<32>(acc); break;
                default: v = group_sum<16>(acc); break;
            }
            if (s == 0 && p < npairs) res[(pc - sl * rpw) * n_slots + sl] = v;
            p += step;
            // (the wave's first lane holds its lowest pair)
            if ((uint32_t)__builtin_amdgcn_readfirstlane((int)p) >= npairs) break;
            i0 = 0;
            acc = 0.0f;
        }
        load(i0);
    }
    // every lane's weight in place before the row branch reads it by lane
    asm volatile("" : "+v"(rw));
    __syncthreads();
    if (tid < nrows) {
        // rank order, one fmaf per slot (the padded sums past n_slots are dropped)
        float y = 0.0f;
#pragma unroll
        for (int k = 0; k < (int)DW_SLOTS; k++) {
            const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rw), k));
            const float v = res[tid * n_slots + k];
            y = k < (int)n_slots ? fmaf(w, v, y) : y;
        }
        a.y[row0 + tid] = y;
    }
    asm volatile("" : "+v"(gen));
    if (a.router && blockIdx.x == 0 && tid == 0) st_dev(a.fsync + 1, gen + 1);
}

template <class QD>
static hipError_t down_wide(const MoeArgs &a, uint32_t n_slots, hipStream_t st) {
    DownPlan p;
    if (!down_plan(QD::TYPE == T_Q6_K, a.hidden, a.ffn, n_slots, (uint32_t)device_cu_count(), p))
        return hipErrorInvalidValue;
    return with_n<dw_nmax<QD>()>(p.N, [&](auto n) -> hipError_t {
        constexpr int N = decltype(n)::value;
        auto kern = p.pack ? k_moe_down_wide<QD, N, true> : k_moe_down_wide<QD, N, false>;
        const hipError_t e = lds_limit(kern, p.lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3((a.hidden + p.rpw - 1) / p.rpw), dim3(64 * p.nw), p.lds, st, a, p.rpw, p.inv_rpw,
                           n_slots, (uint32_t)ilog2(p.S));
        return hipGetLastError();
    });
}

hipError_t launch_moe_down_wide(const MoeArgs &a, uint32_t n_slots, hipStream_t s) {
    return a.down_type == T_Q6_K ? down_wide<Q6K>(a, n_slots, s) : down_wide<Q4K>(a, n_slots, s);
}

// ---------------------------------------------------------------------------
// The grouped down kernel for Q4_K rows above 16 blocks: a workgroup takes
// GL_ROWS output rows of an entry's expert, a wave one row at a time with the
// wide kernel's split (64 lanes, the same items in the same order, so a pair's
// sum has the bits of the single-token layer's), N items per lane and batch,
// the next batch's loads in flight while every pair is dotted with this one's.
// The entry's h is staged once per workgroup, 11 KB a pair at 8192 columns
// against 147 KB of weights in 32 rows. A loop of 8 lanes per row with one
// block in flight took the batched layer of 24 tokens (top-2 of 8, hidden
// 4096) 605 us at ffn 8192 and 1067 at 14336; with this kernel 261 and 440.
// ---------------------------------------------------------------------------
constexpr uint32_t GL_ROWS = 32;
constexpr int GL_NMAX = 4;
constexpr uint32_t GL_MAX_NT = 512;

template <int N>
__global__ void __launch_bounds__(GL_MAX_NT) k_moe_down_grp_long(MoeArgs a) {
    extern __shared__ __align__(16) uint8_t lds[];
    using X = XLds<Q4K, 1>;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockDim.x, nw = nt / WAVE;
    const GrpEntry ent = grp_entry(a, blockIdx.y);
    const uint32_t ex = ent.ex, cnt = ent.cnt;
    if (cnt == 0) return;   // whole workgroup, before any barrier
    const uint32_t nb = a.ffn / 256, items = nb * Q4K::IPB;
    const uint64_t hstride = (uint64_t)(a.ffn / 32) * 36, rb = (uint64_t)nb * Q4K::BB;
    const uint32_t per = a.ffn / 16, ntask = cnt * per;
    auto h_load = [&](uint32_t t) {   // whole waves (the lane exchange)
        const uint32_t g = t / per;
        return dw_load_h(a.hq8 + (uint64_t)(uint32_t)__shfl((int)ent.pair, (int)g, WAVE) * hstride, t - g * per);
    };
    DwH hv[DW_HT];
#pragma unroll
    for (int i = 0; i < DW_HT; i++) hv[i] = h_load(min(tid + nt * i, ntask - 1));   // clamped, not skipped
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t row0 = blockIdx.x * GL_ROWS, nrows = min(GL_ROWS, a.hidden - row0);
    const uint8_t *db = ex >= a.n_expert ? a.down_sh : a.down + (uint64_t)ex * a.hidden * rb;
    typename Q4K::Raw raw[N];
    auto load = [&](uint32_t r, uint32_t i0) {
        const uint8_t *rp = db + (uint64_t)(row0 + min(r, nrows - 1)) * rb;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t item = min(lane + WAVE * (i0 + i), items - 1);
            raw[i] = Q4K::load(rp + (item / Q4K::IPB) * Q4K::BB, (int)(item % Q4K::IPB));
        }
    };
    load(wave, 0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);   // the first weight loads are out before h is staged
#pragma unroll
    for (int i = 0; i < DW_HT; i++)
        if (const uint32_t t = tid + nt * i; t < ntask) dw_put_h<Q4K>(lds, t / per * items, t % per, hv[i]);
    for (uint32_t t0 = nt * DW_HT; t0 < ntask; t0 += nt) {
        const uint32_t t = tid + t0;
        const DwH v = h_load(min(t, ntask - 1));
        if (t < ntask) dw_put_h<Q4K>(lds, t / per * items, t % per, v);
    }
    __syncthreads();   // the last barrier: waves end on their own
    if (wave >= nrows) return;

    float acc[GRP_MAX];
#pragma unroll
    for (uint32_t g = 0; g < GRP_MAX; g++) acc[g] = 0.0f;
    for (uint32_t r = wave, i0 = 0;;) {
        typename Q4K::Raw cur[N];
#pragma unroll
        for (int i = 0; i < N; i++) cur[i] = raw[i];
        const uint32_t base = i0, row = row0 + r;
        i0 += N;
        const bool done = WAVE * i0 >= items;   // this batch ends the row
        if (done) {
            r += nw;
            i0 = 0;
        }
        const bool more = !done || r < nrows;
        if (more) load(r, i0);
#pragma unroll
        for (uint32_t g = 0; g < GRP_MAX; g++) {
            if (g >= cnt) break;   // uniform
#pragma unroll
            for (int i = 0; i < N; i++) {
                const uint32_t at = lane + WAVE * (base + i), item = min(at, items - 1);
                const X x(lds, g * items + item);
                const float v = item_dot<1>(cur[i], (int)(item % Q4K::IPB), x);
                acc[g] += at < items ? v : 0.0f;
            }
            if (done) {
                const float v = group_sum<64>(acc[g]);
                const uint32_t pair = (uint32_t)__builtin_amdgcn_readlane((int)ent.pair, (int)g);
                if (lane == 0) a.yp[(uint64_t)pair * a.hidden + row] = v;
                acc[g] = 0.0f;
            }
        }
        if (!more) break;
    }
}

hipError_t launch_moe_groups_down_long(const MoeArgs &a, uint32_t max_entries, hipStream_t s) {
    const uint32_t nb = a.ffn / 256, items = nb * Q4K::IPB;
    const uint32_t steps = (items + WAVE - 1) / WAVE, batches = (steps + GL_NMAX - 1) / GL_NMAX;
    const uint32_t lds = XLds<Q4K, 1>::bytes(GRP_MAX * items);
    // eight waves where one workgroup fills the LDS of a CU, four of two
    const uint32_t nw = lds > LDS_PER_WG / 2 ? 8 : 4;
    return with_n<GL_NMAX>((steps + batches - 1) / batches, [&](auto n) -> hipError_t {
        auto kern = k_moe_down_grp_long<decltype(n)::value>;
        const hipError_t e = lds_limit(kern, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3((a.hidden + GL_ROWS - 1) / GL_ROWS, max_entries), dim3(64 * nw), lds, s, a);
        return hipGetLastError();
    });
}

}  // namespace kq
