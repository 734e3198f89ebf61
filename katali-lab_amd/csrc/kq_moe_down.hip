// kq_moe_down.hip — kernel B for long down rows (more than four blocks per
// lane at kernel B's own lane counts, or a shape none of its unrolled
// variants takes): weighted down projection of a layer's slots.
//
// A workgroup takes a run of output rows and all their slots, pair (slot, row)
// after pair with the rows of one slot in a row, so it reads each slot's rows
// as one stretch of memory. A pair is dotted by S lanes of a wave (64, or 4
// blocks' items for rows of 5 to 16 blocks), N items each per batch with all
// their loads in flight; every slot's h is staged once per workgroup in item
// order (kq_items.h). The partial sums of a pair meet on the VALU, the rows'
// slots in rank order as in kernel B.
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
constexpr uint32_t DW_SLOTS = 17;   // the most slots of a layer (16 routed and the shared expert)
constexpr int DW_HT = 4;            // h tasks per thread in registers ahead of the weights

template <class QD>
constexpr int dw_nmax() { return QD::TYPE == T_Q4_K ? 8 : 4; }

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
// task t: run t % (ffn / 16) of slot t / (ffn / 16)
template <class QD>
__device__ __forceinline__ void dw_put_h(uint8_t *lds, uint32_t per, uint32_t slot_bytes, uint32_t t, const DwH &h) {
    using X = XLds<QD, 1>;
    uint32_t item, grp;
    X::place(t % per, item, grp);
    const X x(lds + t / per * slot_bytes, item);
    *(uint4 *)x.xq(grp) = h.q;
    int sum = dot4(h.q.x, 0x01010101u, 0);
    sum = dot4(h.q.y, 0x01010101u, sum);
    sum = dot4(h.q.z, 0x01010101u, sum);
    sum = dot4(h.q.w, 0x01010101u, sum);
    *x.isum(grp) = sum;
    if ((t & 1) == 0) *x.d8(grp) = h2f(h.d);   // both halves of a block share it
}

template <class QD, int N>
__global__ void __launch_bounds__(DW_MAX_NT) k_moe_down_wide(MoeArgs a, uint32_t rpw, uint32_t inv_rpw, uint32_t n_slots,
                                                              uint32_t log2s) {
    extern __shared__ __align__(16) uint8_t lds[];
    using X = XLds<QD, 1>;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockDim.x;
    const uint32_t nb = a.ffn / 256, items = nb * QD::IPB, slot_bytes = X::bytes(items);
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
        if (tid + nt * i < ntask) dw_put_h<QD>(lds, per, slot_bytes, tid + nt * i, hv[i]);
    for (uint32_t t = tid + nt * DW_HT; t < ntask; t += nt) dw_put_h<QD>(lds, per, slot_bytes, t, dw_load_h(a.hq8, t));
    __syncthreads();

    float *res = (float *)(lds + n_slots * slot_bytes);   // [row][slot]
    float acc = 0.0f;
    // batches of a pair, then the next pair, in one loop with one load: two
    // loads (or a nested loop) cost a second set of raw registers
    for (uint32_t i0 = 0;;) {
        const uint32_t pc = min(p, npairs - 1), sl = pc * inv_rpw >> 20;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t at = s + S * (i0 + i), item = min(at, items - 1);
            const X x(lds + sl * slot_bytes, item);
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
    const uint32_t nb = a.ffn / 256, items = nb * QD::IPB, cus = (uint32_t)device_cu_count();
    // rows of 5 to 16 blocks: four block columns of lanes (the grouped down
    // kernel's split, whose bits these are); longer rows: the whole wave
    const uint32_t S = nb > 16 ? 64 : 4 * QD::IPB, sp = 64 / S;
    const uint32_t steps = (items + S - 1) / S, nmax = dw_nmax<QD>(), batches = (steps + nmax - 1) / nmax;
    const uint32_t hb = n_slots * XLds<QD, 1>::bytes(items);
    // two workgroups of 8 waves per CU while their h fits twice, else one of
    // 16 waves; never more waves than the rows give pairs
    const uint32_t per_cu = hb + 4096 <= LDS_PER_WG / 2 ? 2 : 1, wmax = per_cu == 2 ? 8 : 16;
    const uint32_t rpw = (a.hidden + per_cu * cus - 1) / (per_cu * cus);
    const uint32_t lds = hb + (rpw * n_slots + DW_SLOTS) * 4;
    if (lds > LDS_PER_WG) return hipErrorNotSupported;
    uint32_t nw = (rpw * n_slots + sp - 1) / sp;
    nw = nw < 4 ? 4 : (nw > wmax ? wmax : nw);
    if (rpw > 64 * nw || rpw > 200) return hipErrorNotSupported;   // a thread per row at the end; inv_rpw exact
    return with_n<dw_nmax<QD>()>((steps + batches - 1) / batches, [&](auto n) -> hipError_t {
        auto kern = k_moe_down_wide<QD, decltype(n)::value>;
        const hipError_t e = lds_limit(kern, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3((a.hidden + rpw - 1) / rpw), dim3(64 * nw), lds, st, a, rpw,
                           ((1u << 20) + rpw - 1) / rpw, n_slots,
                           (uint32_t)ilog2(S));
        return hipGetLastError();
    });
}

hipError_t launch_moe_down_wide(const MoeArgs &a, uint32_t n_slots, hipStream_t s) {
    if (n_slots == 0 || n_slots > DW_SLOTS || a.ffn <= 1024) return hipErrorNotSupported;
    return a.down_type == T_Q6_K ? down_wide<Q6K>(a, n_slots, s) : down_wide<Q4K>(a, n_slots, s);
}

}  // namespace kq
