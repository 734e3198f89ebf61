// kq_plan.h — host-side launch decisions that need no device, shared by the
// launchers and by CPU tests (plain C++, no HIP headers).
#pragma once

#include <stdint.h>

#include <initializer_list>

namespace kq {

// The one-launch layers (the XCD-sliced layer and its stack) wait between
// their workgroups, so all `grid` of them must be resident at once: one per
// CU on a device of exactly `grid` CUs (the slot-to-XCD mapping), with the
// occupancy API's blocks_per_cu for the kernel's block size and LDS at
// least 1.
inline bool xcd_coresident(int cus, int blocks_per_cu, uint32_t grid) {
    return cus > 0 && (uint32_t)cus == grid && blocks_per_cu >= 1 && (uint64_t)blocks_per_cu * (uint64_t)cus >= grid;
}

// Kernel A: units of 32 h values (a q8_1 block) put ceil(units / cus) on the
// busiest CU; half units put ceil(2 units / cus) halves there. Half units when
// that is less work on the busiest CU and the units pair up by eights (384
// units on 256 CUs: 2 against 1.5).
inline bool half_units(uint32_t units, uint32_t cus) {
    if (!cus || units % 8) return false;
    const uint64_t full = (units + cus - 1) / cus, half = (2ull * units + cus - 1) / cus;
    return half < 2 * full;
}

// gfx950's LDS per workgroup
constexpr uint32_t LDS_PER_WG = 160 * 1024;

// The wide down projection's launch (k_moe_down_wide): a workgroup of nw waves
// takes rpw output rows of all slots, S lanes per (slot, row) pair and N items
// per lane and batch. h in item order is 352 bytes per block in tiles of 16
// items, each slot from a tile of its own while that fits, else slot after slot
// (pack): at most 1056 bytes more than the 11/8 per value of the layer's LDS
// rule, which keeps 2116 bytes for the rows' sums, so every shape that rule
// admits has a plan.
constexpr uint32_t DW_SLOTS = 17;       // the most slots of a layer (16 routed and the shared expert)
constexpr uint32_t DW_MAX_ROWS = 200;   // inv_rpw exact, a thread per row at the end
struct DownPlan {
    uint32_t S, N, rpw, inv_rpw, nw, lds;
    bool pack;
};
inline uint32_t item_tile_bytes(uint32_t items, uint32_t ipb) { return (items + 15) / 16 * (16 / ipb * 352); }
inline bool down_plan(bool q6, uint32_t hidden, uint32_t ffn, uint32_t n_slots, uint32_t cus, DownPlan &p) {
    const uint32_t ipb = q6 ? 4 : 8, nb = ffn / 256, items = nb * ipb, nmax = q6 ? 4 : 8;
    if (!cus || nb <= 4 || n_slots == 0 || n_slots > DW_SLOTS) return false;
    // rows of 5 to 16 blocks: four block columns of lanes; longer rows: the
    // whole wave (the grouped down kernels' split)
    p.S = nb > 16 ? 64 : 4 * ipb;
    const uint32_t steps = (items + p.S - 1) / p.S, batches = (steps + nmax - 1) / nmax;
    p.N = (steps + batches - 1) / batches;
    // two workgroups of 8 waves per CU while their h fits twice, with Q4_K up
    // to 7/16 of the LDS (nine slots of 6144: 41.9 us staged twice, 40.5 once),
    // else one of 16 waves; never more waves than the rows give pairs
    uint32_t hb = n_slots * item_tile_bytes(items, ipb);
    const uint32_t per_cu = hb + (q6 ? 4096 : 10240) <= LDS_PER_WG / 2 ? 2 : 1, wmax = per_cu == 2 ? 8 : 16;
    p.rpw = (hidden + per_cu * cus - 1) / (per_cu * cus);
    const uint32_t most_rpw = p.rpw < DW_MAX_ROWS ? p.rpw : DW_MAX_ROWS;
    p.pack = hb + (most_rpw * n_slots + DW_SLOTS) * 4 > LDS_PER_WG;
    if (p.pack) hb = item_tile_bytes(n_slots * items, ipb);
    if (hb + (n_slots + DW_SLOTS) * 4 > LDS_PER_WG) return false;
    const uint32_t fit = ((LDS_PER_WG - hb) / 4 - DW_SLOTS) / n_slots;
    for (uint32_t most : {fit, DW_MAX_ROWS})
        if (p.rpw > most) p.rpw = most;
    p.inv_rpw = ((1u << 20) + p.rpw - 1) / p.rpw;
    p.nw = (p.rpw * n_slots + 64 / p.S - 1) / (64 / p.S);
    p.nw = p.nw < 4 ? 4 : (p.nw > wmax ? wmax : p.nw);
    p.lds = hb + (p.rpw * n_slots + DW_SLOTS) * 4;
    return true;
}

}  // namespace kq
