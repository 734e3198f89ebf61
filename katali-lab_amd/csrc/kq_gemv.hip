// kq_gemv.hip — q8_1 quantization, dense Q4_K / Q6_K GEMV (fp32 and q8_1
// activations), per-block integer sums, synthetic data and a copy kernel.
//
// GEMV layout: a row is nb = cols/256 super-blocks = nb*IPB lane items. S lanes
// (a power of two, at most 64) share a row and each takes N items of it per
// batch (item = s + S*i, so a wave instruction walks consecutive items of a
// row; gemv_shape picks S and N). A wave holds 64/S rows at a time and each
// slot issues the loads of RPS rows, N items each, before it computes any of
// them. The activation is staged once per workgroup in LDS, in item order.
//
// Bound by the weight stream for large matrices (Q6_K 151936 x 2048, q8_1:
// 48.2 us, 5.3 TB/s, before the quad loads 50.6; Q4_K with an fp32 activation
// by its converts and FMAs, about 110 per 18 bytes: 40000 x 5120 4.0 TB/s), by
// launch, first loads and tail below about 20 MB. Row lengths that are no
// power of two used to run a loop over items with one load in flight and as
// few as 4 lanes per row (weights from memory: Q6_K 5120 x 13824, fp32, 50.3 us,
// now 20.1; Q4_K 9731 x 2560, quantizing, 8.9, now 5.6; q, k, v of 2560 columns
// 10.1, now 5.9; weights in the cache, the first two 37.2, now 16.6, and 7.1,
// now 5.2).
#include "kq_device.h"
#include "kq_items.h"
#include "kq_launch.h"

namespace kq {

int device_cu_count() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cached[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}

__global__ void __launch_bounds__(256) k_quantize_q8_1(const float *__restrict__ x, uint32_t nblk,
                                                        uint8_t *__restrict__ out) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nblk * 8) return;   // whole 8-lane groups exit together
    const uint32_t blk = t >> 3, part = t & 7;
    const float4 v = *(const float4 *)(x + 32 * blk + 4 * part);
    uint32_t d16, s16;
    int lo, hi;
    float dd;
    const uint32_t q = quant_q8_1_part(v, d16, s16, lo, hi, dd);
    uint8_t *b = out + 36 * blk;
    *(uint32_t *)(b + 4 + 4 * part) = q;
    if (part == 0) *(uint32_t *)b = d16 | (s16 << 16);
}

hipError_t launch_quantize_q8_1(const float *x, uint64_t n, uint8_t *out, hipStream_t s) {
    const uint32_t nblk = (uint32_t)(n / 32);
    const uint32_t threads = nblk * 8;
    hipLaunchKernelGGL(k_quantize_q8_1, dim3((threads + 255) / 256), dim3(256), 0, s, x, nblk, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// GEMV
// ---------------------------------------------------------------------------
// Rows a lane slot loads together, by the items each lane takes of a row, and
// the most items per batch (Q4_K: 8 VGPRs of raw block each, Q6_K: 14).
template <class QT>
constexpr int gemv_rps(int n) {
    return QT::TYPE == T_Q4_K ? (n == 1 ? 4 : (n == 2 ? 2 : 1)) : (n == 1 ? 2 : 1);
}
template <class QT>
constexpr int gemv_nmax() { return QT::TYPE == T_Q4_K ? 8 : 5; }
constexpr int GEMV_MAX_NT = 512;
constexpr uint32_t GEMV_MAX_COLS = 32768;

// The activation, staged in two halves around the weight loads: load() issues
// the first XPRE tasks per thread into registers (the whole activation for
// cols <= 4096 in 256 threads), store() writes them to LDS after the weight
// loads are out and stages any remaining tasks directly. A task is 4 values:
// fp32 copied (MODE 0), q8_1 bytes copied (MODE 1), or fp32 quantized to q8_1
// with 8 lanes per block (MODE 2).
constexpr int XPRE = 4;
template <class QT, int MODE>
struct XStage {
    using X = XLds<QT, MODE>;
    float4 v[XPRE];
    uint32_t q[XPRE], d[XPRE];
    __device__ __forceinline__ void load(const float *xf, const uint8_t *xq, uint32_t cols) {
        const uint32_t n = cols / 4, nt = blockDim.x;
#pragma unroll
        for (int i = 0; i < XPRE; i++) {
            if (nt * i >= n) break;                                // uniform
            const uint32_t t = min(threadIdx.x + nt * i, n - 1);   // clamped, not skipped
            if constexpr (MODE == 1) {
                const uint8_t *b = xq + (t >> 3) * 36;
                q[i] = *(const uint32_t *)(b + 4 + 4 * (t & 7));
                d[i] = ld_u16(b);
                v[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            } else {
                v[i] = *(const float4 *)(xf + 4 * t);
                q[i] = d[i] = 0;
            }
        }
    }
    __device__ __forceinline__ void put(uint32_t t, float4 x4, uint32_t qq, uint32_t dd, uint8_t *lds) const {
        uint32_t item, grp;
        X::place(t >> 2, item, grp);
        const X x(lds, item);
        if constexpr (MODE == 0) {
            *x.xf(4 * grp + (t & 3)) = x4;
        } else {
            uint32_t qv;
            int lo, hi;
            float dec;
            if constexpr (MODE == 1) {
                qv = qq;
                q8_part_sums(qv, lo, hi);
                dec = h2f(dd);
            } else {
                uint32_t d16, s16;
                qv = quant_q8_1_part(x4, d16, s16, lo, hi, dec);
            }
            ((uint32_t *)x.xq(grp))[t & 3] = qv;
            if ((t & 3) == 0) {   // parts 0 and 4 of the block: its two halves, one item each
                *x.isum(grp) = (t & 4) ? hi : lo;
                *x.d8(grp) = dec;
            }
        }
    }
    // Tasks past n were loaded clamped and are dropped here (whole 8-lane
    // groups: n % 8 == 0); the barriers around the weight loads keep the
    // compiler from sinking the preloads into these branches.
    __device__ __forceinline__ void store(const float *xf, const uint8_t *xq, uint32_t cols, uint8_t *lds) const {
        const uint32_t n = cols / 4, nt = blockDim.x;
#pragma unroll
        for (int i = 0; i < XPRE; i++) {
            const uint32_t t = threadIdx.x + nt * i;
            if (t < n) put(t, v[i], q[i], d[i], lds);
        }
        for (uint32_t t = threadIdx.x + nt * XPRE; t < n; t += nt) {   // whole 8-lane groups (n % 8 == 0)
            float4 x4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            uint32_t qq = 0, dd = 0;
            if constexpr (MODE == 1) {
                const uint8_t *b = xq + (t >> 3) * 36;
                qq = *(const uint32_t *)(b + 4 + 4 * (t & 7));
                dd = ld_u16(b);
            } else {
                x4 = *(const float4 *)(xf + 4 * t);
            }
            put(t, x4, qq, dd, lds);
        }
        if constexpr (MODE == 0) {   // half-block sums of the fp32 activation
            __syncthreads();
            for (uint32_t h = threadIdx.x; h < cols / 16; h += nt) {
                uint32_t item, grp;
                X::place(h, item, grp);
                const X x(lds, item);
                float sum = 0.0f;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 w = *x.xf(4 * grp + j);
                    sum += w.x;
                    sum += w.y;
                    sum += w.z;
                    sum += w.w;
                }
                *x.fsum(grp) = sum;
            }
        }
    }
};

// The row groups of one matrix that workgroup `block` of `nblocks` takes
// (the workgroups' shares of the matrix interleave: a grid-stride loop). The
// S lanes of a row take items s, s + S, ... in batches of N, all of a batch's
// loads in flight at once; items past the row's end load the last one and
// count as zero.
// SPAN: 64, a row takes the whole wave; 32, at most half of it; 0, either. A
// kernel with both ways to sum a row costs a call of a few microseconds 0.05
// to 0.2 us (quantizing, Q4_K 512 x 256: 2.73 us, apart 2.51; 2048 x 2048: 3.14
// and 3.00); the launch of several matrices, which may hold both, loses with
// kernels of their own (q, k and v of 4096 columns 6.7 -> 6.9 us).
template <class QT, int N, int RPS, int MODE, int SPAN, bool PIN = false>
__device__ __forceinline__ void gemv_rows(const uint8_t *__restrict__ w, uint32_t rows, uint32_t cols, uint64_t rb,
                                          uint32_t log2s, const float *xf, const uint8_t *xq, float *__restrict__ y,
                                          uint32_t block, uint32_t nblocks, uint8_t *lds) {
    if constexpr (SPAN == 64) log2s = 6;
    const uint32_t S = 1u << log2s;
    const uint32_t slots = WAVE >> log2s;
    const uint32_t lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE, NW = blockDim.x / WAVE;
    const uint32_t slot = lane >> log2s, s = lane & (S - 1);
    const uint32_t items = cols / 256 * QT::IPB;
    const uint32_t rows_iter = NW * slots * RPS;
    const uint32_t base0 = block * rows_iter;
    auto row_of = [&](uint32_t base, int r) { return base + r * (NW * slots) + wave * slots + slot; };

    // The activation loads, then the first row group's weight loads, go out
    // before the activation is staged, so the two latencies overlap. Rows are
    // clamped, not skipped (a load under a branch makes the compiler wait for
    // all).
    typename QT::RawQ raw[RPS][N];   // (a quad's lanes hold one block's items, or all lie past the row)
    auto load_rows = [&](uint32_t base, uint32_t i0) {
#pragma unroll
        for (int r = 0; r < RPS; r++) {
            const uint8_t *rp = w + (uint64_t)min(row_of(base, r), rows - 1) * rb;
#pragma unroll
            for (int i = 0; i < N; i++) {
                const uint32_t item = min(s + S * (i0 + i), items - 1);
                raw[r][i] = QT::load_quad(rp + (item / QT::IPB) * QT::BB, item % QT::IPB);
            }
        }
    };
    // The matrix's arguments with x's, not in a second round trip behind x's
    // loads (gemv_multi_pin; one matrix's arguments are one cache line).
    if constexpr (PIN) pin_args(w, rows, rb, log2s, nblocks);
    XStage<QT, MODE> xs;
    xs.load(xf, xq, cols);   // issued first: waiting for x then waits for nothing else
    // Neither the compiler nor the scheduler may move work across these two
    // points (x is deliberately not __restrict__, so its loads are not
    // treated as invariant and re-issued at their use).
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    load_rows(base0, 0);   // base0 < rows: the grid never exceeds the row groups
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);   // every weight load is out before x is staged
    xs.store(xf, xq, cols, lds);
    __syncthreads();

    float acc[RPS];
#pragma unroll
    for (int r = 0; r < RPS; r++) acc[r] = 0.0f;
    for (uint32_t base = base0, i0 = 0;;) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t at = s + S * (i0 + i), item = min(at, items - 1);
            const XLds<QT, MODE> x(lds, item);
#pragma unroll
            for (int r = 0; r < RPS; r++) {
                const float v = item_dot<MODE>(QT::full(raw[r][i]), item % QT::IPB, x);
                acc[r] += at < items ? v : 0.0f;
            }
            // The rows share an item's activation; the next item's is read
            // when this one's dots are done (left alone, the compiler reads
            // every item's first and keeps them in registers, or spills).
#pragma unroll
            for (int r = 0; r < RPS; r++) asm volatile("" : "+v"(acc[r])::"memory");
        }
        i0 += N;
        if (S * i0 >= items) {   // the row group is done
            if (SPAN == 64 || (SPAN == 0 && log2s == 6)) {
                // one row per wave instruction: the RPS rows reduce together
                // (halving exchanges, no LDS); lane groups of 64 / RPS then
                // hold row (lane >> SH) & (RPS - 1)
                constexpr int LOGR = RPS >= 4 ? 2 : (RPS >= 2 ? 1 : 0);
                constexpr int SH = 6 - LOGR;
                const float v = reduce_rows<RPS>(acc);
                const uint32_t r = (lane >> SH) & (RPS - 1);
                const uint32_t row = row_of(base, (int)r);
                if ((lane & ((1u << SH) - 1)) == 0 && row < rows) y[row] = v;
            } else if constexpr (SPAN == 32) {
                auto sums = [&](auto g) {   // the lanes of a row slot sum on the VALU
#pragma unroll
                    for (int r = 0; r < RPS; r++) acc[r] = group_sum<decltype(g)::value>(acc[r]);
                };
                switch (log2s) {   // uniform
                    case 5: sums(std::integral_constant<int, 32>{}); break;
                    case 4: sums(std::integral_constant<int, 16>{}); break;
                    case 3: sums(std::integral_constant<int, 8>{}); break;
                    default: sums(std::integral_constant<int, 4>{}); break;
                }
#pragma unroll
                for (int r = 0; r < RPS; r++) {
                    const uint32_t row = row_of(base, r);
                    if (s == 0 && row < rows) y[row] = acc[r];
                }
            } else {
#pragma unroll
                for (int r = 0; r < RPS; r++) {
                    float v;
                    switch (log2s) {   // uniform
                        case 5: v = group_sum<32>(acc[r]); break;
                        case 4: v = group_sum<16>(acc[r]); break;
                        case 3: v = group_sum<8>(acc[r]); break;
                        default: v = group_sum<4>(acc[r]); break;
                    }
                    const uint32_t row = row_of(base, r);
                    if (s == 0 && row < rows) y[row] = v;
                }
            }
            base += nblocks * rows_iter;
            if (base >= rows) break;
            i0 = 0;
#pragma unroll
            for (int r = 0; r < RPS; r++) acc[r] = 0.0f;
        }
        load_rows(base, i0);
    }
}

template <class QT, int N, int RPS, int MODE, int SPAN>
__global__ void __launch_bounds__(GEMV_MAX_NT)
    k_gemv(const uint8_t *__restrict__ w, uint32_t rows, uint32_t cols, uint64_t rb, uint32_t log2s,
           const float *xf, const uint8_t *xq, float *__restrict__ y) {
    extern __shared__ __align__(16) uint8_t lds[];
    gemv_rows<QT, N, RPS, MODE, SPAN>(w, rows, cols, rb, log2s, xf, xq, y, blockIdx.x, gridDim.x, lds);
}

// Where the launch of several matrices reads a matrix's arguments ahead of x's
// loads: up to 2048 columns and quantizing up to 4096, by Q4_K's items a lane
// (weights from memory, without and with: quantizing, q, k and v of 512 columns
// 3.39 -> 3.32 us, of 4096 6.75 -> 6.70). For longer rows x's loads behind one
// more wait cost what it gains or more (fp32 4096 6.72 and 6.76, quantizing 3072
// 5.66 and 5.72).
template <int N4, int MODE>
constexpr bool gemv_multi_pin() { return N4 == 1 || (MODE == 2 && N4 == 2); }

// Up to four GEMVs over one activation in one launch (the engine's
// matvec_multi: q, k and v of a layer). Matrix m owns workgroups
// [end[m-1], end[m]) and runs the single-matrix body on them, so each row's
// arithmetic, and its bits, are those of k_gemv.
template <int N4, int N6, int MODE>
__global__ void __launch_bounds__(GEMV_MAX_NT) k_gemv_multi(GemvMultiArgs g) {
    extern __shared__ __align__(16) uint8_t lds[];
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < GEMV_MULTI_MAX - 1; i++)
        if (blockIdx.x >= g.end[i]) m = i + 1;   // end[] is non-decreasing, padded with the total
    const uint32_t start = m ? g.end[m - 1] : 0;
    const uint32_t blk = blockIdx.x - start, nblk = g.end[m] - start;
    constexpr bool PIN = gemv_multi_pin<N4, MODE>();
    if (g.type[m] == T_Q4_K)
        gemv_rows<Q4K, N4, gemv_rps<Q4K>(N4), MODE, 0, PIN>(g.w[m], g.rows[m], g.cols,
                                                            (uint64_t)(g.cols / 256) * Q4K::BB, g.log2s[m], g.x, nullptr,
                                                            g.y[m], blk, nblk, lds);
    else
        gemv_rows<Q6K, N6, gemv_rps<Q6K>(N6), MODE, 0, PIN>(g.w[m], g.rows[m], g.cols,
                                                            (uint64_t)(g.cols / 256) * Q6K::BB, g.log2s[m], g.x, nullptr,
                                                            g.y[m], blk, nblk, lds);
}

// How a row's items are spread: S lanes (a power of two) take N items each
// per batch. The widest S that takes the row in one batch (any batches for 64
// lanes: rows past every S) and pads it by at most a quarter (items past the
// row's end, computed and dropped), else by at most a third, else a half:
// wide rows read longer runs per instruction, and leave a lane fewer items in
// a chain and a small matrix more waves (Q4_K 9731 x 2560, 32 lanes x 3
// items: 5.6 us, 16 x 5: 6.4; 5120 x 5120 6.5 and 7.7). A large matrix fills
// the chip either way and pays for the padding instead, so there at most an
// eighth comes first (q8_1 and weights from memory: Q4_K 20000 x 5120, 64 x 3:
// 13.7 us, 32 x 5: 12.5; Q6_K 40000 x 5120 35.7 and 33.2).
struct GemvShape {
    uint32_t S, N;
};
constexpr GemvShape gemv_shape(uint32_t items, uint32_t nmax, bool large) {
    for (uint32_t den = large ? 8 : 4; den >= 2; den = den == 8 ? 4 : den - 1)
        for (uint32_t S = 64; S >= 4; S >>= 1) {
            const uint32_t steps = (items + S - 1) / S, batches = (steps + nmax - 1) / nmax;
            const uint32_t N = (steps + batches - 1) / batches;
            if ((batches == 1 || S == 64) && den * S * N * batches <= (den + 1) * items) return {S, N};
        }
    return {64, nmax};
}
// The shapes of every row length, formed at compile time: gemv_pair picks the
// kernels of several matrices from them (a launch saves 13 ns of divisions on
// average, 55 at most).
struct GemvShapes {
    GemvShape s[GEMV_MAX_COLS / 256 + 1][2];
};
template <class QT>
constexpr GemvShapes gemv_shapes() {
    GemvShapes t{};
    for (uint32_t nb = 1; nb <= GEMV_MAX_COLS / 256; nb++)
        for (int l = 0; l < 2; l++) t.s[nb][l] = gemv_shape(nb * QT::IPB, gemv_nmax<QT>(), l != 0);
    return t;
}
template <class QT>
inline constexpr GemvShapes GEMV_SHAPES = gemv_shapes<QT>();
// large: from 10240 items per CU, 2.6 million (the least padded spread loses
// up to 2.2 million, Q4_K 18944 x 3584 10.6 against 9.3 us, Q6_K 20000 x 5120
// 20.8 against 19.8, 28000 x 5120 26.6 against 25.8, and wins from 3.2 million);
// from 6144, 1.6 million, with Q6_K up to 4096 columns, whose least padded rows
// run in workgroups of 4 waves (gemv_grid; 40000 x 2560 18.2 against 19.7).
template <class QT>
constexpr GemvShape gemv_shape(uint64_t rows, uint64_t cols, uint64_t cus) {
    const uint64_t nb = cols / 256, line = QT::TYPE == T_Q6_K && cols <= 4096 ? 6144 : 10240;
    return GEMV_SHAPES<QT>.s[nb][rows * nb * QT::IPB > line * cus];
}
// the item counts that the two formats have at one and the same row length
constexpr bool gemv_pair(uint32_t n4, uint32_t n6) {
    for (uint64_t nb = 1; nb <= GEMV_MAX_COLS / 256; nb++)
        if (GEMV_SHAPES<Q4K>.s[nb][0].N == n4 && GEMV_SHAPES<Q6K>.s[nb][0].N == n6) return true;
    return false;
}

// Waves per workgroup and the most workgroups per CU, for `waves` waves of
// rows; the busiest CU, with the most of them, sets the time. us with q8_1 and
// weights from memory where nothing else is said:
//   - up to 4 waves per CU 4 (no count puts fewer on a CU);
//   - up to 16 the count (4, 6 or 8) that puts the fewest on the busiest CU.
//     Among equals 8 (fewer workgroups stage the activation: Q4_K 4096 x 4096
//     4.3 in 256 workgroups of 8 waves, 4.9 in 512 of 4), but 4 rather than 6 up
//     to 4096 columns, quantizing up to 2048 (Q4_K 6144 x 4096 5.0 and 5.5,
//     11008 x 2048 4.6 and 5.1), and 4 rather than 8 for Q6_K from 2048 to 4096
//     columns and up to 14 waves (14336 x 2560 9.1 and 9.5);
//   - above, workgroups that loop over their rows: two of 8 waves, so that the
//     activation is staged twice per CU rather than once per 4 waves (Q6_K 5120
//     x 13824, fp32: 20.3 against 26.0; Q4_K 9731 x 2560: 6.0 against 6.8), and
//     up to 2048 columns as many of 4 as fit (Q4_K 25000 x 1536: 6.5 against
//     7.1), unless they quantize for Q4_K in more than one round (40000 x 2048:
//     9.5 in two of 8, 11.1). With Q6_K up to 4096 columns and 32 waves
//     (quantizing 20) of 4 too where the busiest CU gets fewer (20000 x 2560:
//     11.0 and 12.6), of batches of five items four (their registers);
//   - past 64 waves per CU each loops many times and four of 8 waves keep more
//     loads in flight (Q4_K 40000 x 4096, fp32: 22.9 against 23.5 in two).
// One of 8 waves, which stages the activation once, where that is most of a
// workgroup's work: quantizing for Q4_K rows of a whole wave from 8 to 16 waves
// per CU (6144 x 4096: 5.5, in two of 6 waves 6.2), and Q6_K rows of four items a
// lane and more from 8 to 32, but not with fp32 (4096 x 14336: 14.0 and 15.7).
struct GemvGrid {
    uint32_t nw, cap;
};
template <class QT, int MODE>
static GemvGrid gemv_grid(GemvShape sh, uint64_t waves, uint64_t cols, uint32_t cus) {
    constexpr bool Q6 = QT::TYPE == T_Q6_K, QUANT = MODE == 2;
    auto upto = [&](uint64_t per_cu) { return waves <= per_cu * cus; };
    auto busiest = [&](uint32_t nw) { return ((waves + nw - 1) / nw + cus - 1) / cus * nw; };
    if (upto(4)) return {4, 8};
    if (!upto(64)) return {8, 4};
    if (sh.S == 64 && !upto(8)) {
        if (Q6 && MODE != 0 && sh.N >= 4 && upto(32)) return {8, 1};
        if (!Q6 && QUANT && cols > 2048 && upto(16)) return {8, 1};
    }
    const uint64_t b4 = busiest(4), b6 = busiest(6), b8 = busiest(8);
    if (upto(16)) {
        const bool four = b4 <= b6 && b4 <= b8 && !upto(8) && cols <= (QUANT ? 2048 : 4096);
        if (four && (b4 < b8 || (Q6 && cols > 2048 && upto(14)))) return {4, 8};
        return b8 <= b4 && b8 <= b6 ? GemvGrid{8, 2} : (b6 <= b4 ? GemvGrid{6, 3} : GemvGrid{4, 8});
    }
    if (cols <= 2048) return !Q6 && QUANT && !upto(32) && b4 >= b8 ? GemvGrid{8, 2} : GemvGrid{4, 8};
    if (Q6 && cols <= 4096) {
        if (sh.N == 5 && upto(32)) return {4, 4};
        if (b4 < b8 && upto(QUANT ? 20 : 32)) return {4, 8};
    }
    return {8, 2};
}

// No more workgroups per CU than their activation leaves room for: an fp32 one
// takes 4.75 bytes a column, from 16640 columns more than half of the LDS, and
// the second half of the grid would queue and stage it again (weights from
// memory, Q6_K 4096 x 16640 22.8 against 18.3 us, Q4_K 8192 x 28672 42.4
// against 36.6).
static GemvGrid lds_fit(GemvGrid g, uint32_t lds) {
    const uint32_t most = LDS_PER_WG / lds;
    if (g.cap > most) g.cap = most;
    return g;
}

template <class QT, int MODE>
static hipError_t gemv_dispatch(const uint8_t *w, uint64_t rows, uint64_t cols, const float *xf, const uint8_t *xq,
                                float *y, hipStream_t st) {
    const int cus = device_cu_count();
    const GemvShape sh = gemv_shape<QT>(rows, cols, (uint64_t)cus);
    const uint64_t rb = cols / 256 * QT::BB;
    const uint32_t lds = XLds<QT, MODE>::bytes((uint32_t)(cols / 256) * QT::IPB);
    return with_n<gemv_nmax<QT>()>(sh.N, [&](auto n) -> hipError_t {
        constexpr int N = decltype(n)::value, RPS = gemv_rps<QT>(N);
        const uint32_t rows_per_wave = 64 / sh.S * RPS;
        const uint64_t waves = (rows + rows_per_wave - 1) / rows_per_wave;
        const GemvGrid gg = lds_fit(gemv_grid<QT, MODE>(sh, waves, cols, cus), lds);
        const uint64_t iters = (waves + gg.nw - 1) / gg.nw, cap = (uint64_t)gg.cap * cus;
        const uint32_t grid = (uint32_t)(iters < cap ? iters : cap);
        auto kern = sh.S == 64 ? k_gemv<QT, N, RPS, MODE, 64> : k_gemv<QT, N, RPS, MODE, 32>;
        const hipError_t e = lds_limit(kern, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * gg.nw), lds, st, w, (uint32_t)rows, (uint32_t)cols, rb,
                           (uint32_t)ilog2(sh.S), xf, xq, y);
        return hipGetLastError();
    });
}

template <int MODE>
static hipError_t gemv_multi_dispatch(GemvMultiArgs &g, int n, const uint64_t *rows, hipStream_t st) {
    // N by the row length alone (one kernel for all the matrices); S per
    // matrix as the single GEMV takes it: a row's bits depend on S only
    const GemvShape s4 = gemv_shape<Q4K>(0, g.cols, 1), s6 = gemv_shape<Q6K>(0, g.cols, 1);
    const uint32_t nb = g.cols / 256, cus = (uint32_t)device_cu_count();
    uint64_t iters[GEMV_MULTI_MAX] = {0}, total = 0;
    uint32_t lds = 0;
    for (int i = 0; i < n; i++) {
        const bool q4 = g.type[i] == T_Q4_K;
        const uint32_t S = q4 ? gemv_shape<Q4K>(rows[i], g.cols, cus).S : gemv_shape<Q6K>(rows[i], g.cols, cus).S;
        const uint32_t rows_per_wave = 64 / S * (q4 ? gemv_rps<Q4K>(s4.N) : gemv_rps<Q6K>(s6.N));
        g.log2s[i] = (uint32_t)ilog2(S);
        iters[i] = (rows[i] + rows_per_wave - 1) / rows_per_wave;
        total += iters[i];
        const uint32_t b = q4 ? XLds<Q4K, MODE>::bytes(nb * Q4K::IPB) : XLds<Q6K, MODE>::bytes(nb * Q6K::IPB);
        if (rows[i] && b > lds) lds = b;
    }
    if (!total) return hipSuccess;
    // The matrices' workgroups differ in work, and small ones even that out:
    // q, k and v of 4096 columns take 6.6 us in 4 waves, 8.3 in 6, 7.6 in 8.
    GemvGrid gg{4, 8};
    if (total > 64ull * cus) gg = {8, 4};
    else if (total > 16ull * cus && g.cols > 2048) gg = {8, 2};
    // From 16 to 64 waves per CU and up to 5120 columns: the workgroups whose
    // last round leaves the busiest CU the fewest waves, the fewest workgroups
    // among equals (quantizing, q, k and v of 4096 rows and columns: 768
    // workgroups of 8 waves are three per CU, 9.1 us, and a round and a half of
    // two per CU, 10.4; of 5120: 6 waves, three per CU, 16.6 and 18.8), but
    // quantizing three per CU rather than two (4096 rows of 5120 columns 13.9
    // and 15.3). At 6144 columns the third staging of the activation costs what
    // it gains (Q4_K, 6144 and twice 1536 rows 11.2 against 10.2 us).
    if (total > 16ull * cus && total <= 64ull * cus && g.cols > 2048 && g.cols <= 5120) {
        uint64_t best = ~0ull;
        for (const GemvGrid c : {GemvGrid{8, MODE == 2 ? 3u : 2u}, GemvGrid{8, 2}, GemvGrid{6, 3}, GemvGrid{8, 4}}) {
            const uint64_t wgs = (total + c.nw - 1) / c.nw, slots = (uint64_t)c.cap * cus;
            const uint64_t busiest = c.nw * (wgs <= slots ? (wgs + cus - 1) / cus : c.cap * ((wgs + slots - 1) / slots));
            if (busiest < best) gg = c, best = busiest;
        }
    }
    total = 0;
    for (int i = 0; i < n; i++) {   // waves -> workgroups
        iters[i] = (iters[i] + gg.nw - 1) / gg.nw;
        total += iters[i];
    }
    const uint64_t cap = (uint64_t)lds_fit(gg, lds).cap * cus;
    uint32_t end = 0;
    for (int i = 0; i < GEMV_MULTI_MAX; i++) {
        if (i < n) {
            uint64_t wg = iters[i];
            if (total > cap && wg) {   // share the capped grid in proportion, at least one each
                wg = wg * cap / total;
                if (!wg) wg = 1;
            }
            end += (uint32_t)wg;
        }
        g.end[i] = end;   // past n: the total, so no workgroup maps there
    }
    return with_n<gemv_nmax<Q4K>()>(s4.N, [&](auto n4) {
        return with_n<gemv_nmax<Q6K>()>(s6.N, [&](auto n6) -> hipError_t {
            constexpr int N4 = decltype(n4)::value, N6 = decltype(n6)::value;
            if constexpr (!gemv_pair(N4, N6)) {
                return hipErrorInvalidValue;
            } else {
                auto kern = k_gemv_multi<N4, N6, MODE>;
                const hipError_t e = lds_limit(kern, lds);
                if (e != hipSuccess) return e;
                hipLaunchKernelGGL(kern, dim3(end), dim3(64 * gg.nw), lds, st, g);
                return hipGetLastError();
            }
        });
    });
}

hipError_t launch_gemv_multi(int n, const uint32_t *types, const uint8_t *const *ws, const uint64_t *rows,
                             uint64_t cols, const float *x, float *const *ys, int mode, hipStream_t st) {
    GemvMultiArgs g{};
    for (int i = 0; i < n; i++) {
        g.w[i] = ws[i];
        g.y[i] = ys[i];
        g.rows[i] = (uint32_t)rows[i];
        g.type[i] = types[i];
    }
    g.cols = (uint32_t)cols;
    g.x = x;
    return mode == 0 ? gemv_multi_dispatch<0>(g, n, rows, st) : gemv_multi_dispatch<2>(g, n, rows, st);
}

hipError_t launch_gemv(uint32_t type, const uint8_t *w, uint64_t rows, uint64_t cols, const float *xf,
                       const uint8_t *xq, float *y, int mode, hipStream_t s) {
    if (type == T_Q4_K) {
        if (mode == 0) return gemv_dispatch<Q4K, 0>(w, rows, cols, xf, xq, y, s);
        if (mode == 1) return gemv_dispatch<Q4K, 1>(w, rows, cols, xf, xq, y, s);
        return gemv_dispatch<Q4K, 2>(w, rows, cols, xf, xq, y, s);
    }
    if (mode == 0) return gemv_dispatch<Q6K, 0>(w, rows, cols, xf, xq, y, s);
    if (mode == 1) return gemv_dispatch<Q6K, 1>(w, rows, cols, xf, xq, y, s);
    return gemv_dispatch<Q6K, 2>(w, rows, cols, xf, xq, y, s);
}

// ---------------------------------------------------------------------------
// Per-block integer sums through the same item routines the GEMV uses.
// One thread per (row, block, item pair) for Q4_K (two half-items summed), one
// per (row, block, item) for Q6_K.
// ---------------------------------------------------------------------------
template <class QT>
__global__ void __launch_bounds__(256) k_isums(const uint8_t *__restrict__ w, uint32_t rows, uint32_t cols,
                                               const uint8_t *__restrict__ xq, int32_t *__restrict__ out) {
    extern __shared__ __align__(16) uint8_t lds[];
    Act a = act_carve(lds, cols);
    act_stage_from_q8(xq, cols, a);
    __syncthreads();
    const uint32_t nb = cols / 256;
    const uint64_t rb = (uint64_t)nb * QT::BB;
    constexpr uint32_t per_blk = QT::TYPE == T_Q4_K ? 4 : 4;   // threads per block
    const uint64_t total = (uint64_t)rows * nb * per_blk;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t c = (uint32_t)(t % per_blk);
        const uint64_t rbk = t / per_blk;
        const uint32_t b = (uint32_t)(rbk % nb);
        const uint64_t row = rbk / nb;
        const uint8_t *blk = w + row * rb + (uint64_t)b * QT::BB;
        if constexpr (QT::TYPE == T_Q4_K) {
            // group g = c: items 2g (hh=0) and 2g+1 (hh=1) cover sub-blocks 2g, 2g+1
            int l0, h0, l1, h1;
            Q4K::isums(Q4K::load(blk, 2 * c), 2 * c, a.qs + 256 * b, l0, h0);
            Q4K::isums(Q4K::load(blk, 2 * c + 1), 2 * c + 1, a.qs + 256 * b, l1, h1);
            int32_t *o = out + row * (cols / 32) + 8 * b + 2 * c;
            o[0] = l0 + l1;
            o[1] = h0 + h1;
        } else {
            int s4[4];
            Q6K::isums(Q6K::load(blk, c), c, a, b, s4);
            const int n = c >> 1, k = c & 1;
            int32_t *o = out + row * (cols / 16) + 16 * b + 8 * n + k;
            for (int tq = 0; tq < 4; tq++) o[2 * tq] = s4[tq];
        }
    }
}

hipError_t launch_isums(uint32_t type, const uint8_t *w, uint64_t rows, uint64_t cols, const uint8_t *xq,
                        int32_t *out, hipStream_t s) {
    const uint64_t total = rows * (cols / 256) * 4;
    uint64_t grid = (total + 255) / 256;
    if (grid > 4096) grid = 4096;
    const uint32_t lds = act_bytes((uint32_t)cols);
    if (type == T_Q4_K)
        hipLaunchKernelGGL(k_isums<Q4K>, dim3((uint32_t)grid), dim3(256), lds, s, w, (uint32_t)rows, (uint32_t)cols,
                           xq, out);
    else
        hipLaunchKernelGGL(k_isums<Q6K>, dim3((uint32_t)grid), dim3(256), lds, s, w, (uint32_t)rows, (uint32_t)cols,
                           xq, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Synthetic data: counter-based splitmix64 stream, one 64-bit draw per 8 bytes.
// Scale fields get |N(0, sigma)| (Box-Muller) encoded as f16.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ float u01(uint64_t r) { return ((float)(r >> 40) + 0.5f) * (1.0f / 16777216.0f); }
__device__ __forceinline__ float halfnormal(uint64_t key, float sigma) {
    const uint64_t r = splitmix64(key);
    const float u1 = u01(r), u2 = u01(splitmix64(r ^ 0x5DEECE66Dull));
    return fabsf(sigma * sqrtf(-2.0f * logf(u1)) * cosf(6.28318530718f * u2));
}

__global__ void __launch_bounds__(256) k_synth_blocks(uint32_t type, uint8_t *__restrict__ dst, uint64_t nblocks,
                                                      uint64_t seed, float sigma) {
    const uint32_t bb = type == T_Q4_K ? 144 : 210;
    const uint64_t total = nblocks * bb;
    const uint64_t nwords = (total + 7) / 8;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nwords; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t r = splitmix64(seed * 0x2545F4914F6CDD1Dull + i);
        const uint64_t off = i * 8;
        if (off + 8 <= total && (off & 7) == 0 && ((uintptr_t)dst & 7) == 0) {
            *(uint64_t *)(dst + off) = r;
        } else {
            for (int k = 0; k < 8 && off + k < total; k++) dst[off + k] = (uint8_t)(r >> (8 * k));
        }
    }
}

__global__ void __launch_bounds__(256) k_synth_scales(uint32_t type, uint8_t *__restrict__ dst, uint64_t nblocks,
                                                      uint64_t seed, float sigma) {
    for (uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; b < nblocks; b += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t key = (seed ^ 0xA0761D6478BD642Full) * 0x9E3779B97F4A7C15ull + 2 * b;
        if (type == T_Q4_K) {
            uint8_t *blk = dst + b * 144;
            const uint32_t d = f2h_rne(halfnormal(key, sigma)), m = f2h_rne(halfnormal(key + 1, sigma));
            blk[0] = (uint8_t)d; blk[1] = (uint8_t)(d >> 8);
            blk[2] = (uint8_t)m; blk[3] = (uint8_t)(m >> 8);
        } else {
            uint8_t *blk = dst + b * 210;
            const uint32_t d = f2h_rne(halfnormal(key, sigma));
            blk[208] = (uint8_t)d; blk[209] = (uint8_t)(d >> 8);
        }
    }
}

hipError_t launch_synth_blocks(uint32_t type, uint8_t *dst, uint64_t nblocks, uint64_t seed, float sigma,
                               hipStream_t s) {
    const uint32_t bb = type == T_Q4_K ? 144 : 210;
    const uint64_t nwords = (nblocks * bb + 7) / 8;
    uint64_t grid = (nwords + 255) / 256;
    if (grid > 16384) grid = 16384;
    hipLaunchKernelGGL(k_synth_blocks, dim3((uint32_t)grid), dim3(256), 0, s, type, dst, nblocks, seed, sigma);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    uint64_t g2 = (nblocks + 255) / 256;
    if (g2 > 16384) g2 = 16384;
    hipLaunchKernelGGL(k_synth_scales, dim3((uint32_t)g2), dim3(256), 0, s, type, dst, nblocks, seed, sigma);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) k_synth_normal(float *__restrict__ dst, uint64_t n, uint64_t seed, float sigma) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t r = splitmix64(seed * 0xD1B54A32D192ED03ull + i);
        const float u1 = u01(r), u2 = u01(splitmix64(r ^ 0x5DEECE66Dull));
        dst[i] = sigma * sqrtf(-2.0f * logf(u1)) * cosf(6.28318530718f * u2);
    }
}

hipError_t launch_synth_normal(float *dst, uint64_t n, uint64_t seed, float sigma, hipStream_t s) {
    uint64_t grid = (n + 255) / 256;
    if (grid > 16384) grid = 16384;
    hipLaunchKernelGGL(k_synth_normal, dim3((uint32_t)grid), dim3(256), 0, s, dst, n, seed, sigma);
    return hipGetLastError();
}

__global__ void k_step_advance(int32_t *step, int32_t n) {
    if (threadIdx.x == 0) {
        const int32_t v = *step + 1;
        *step = v >= n ? 0 : v;
    }
}

hipError_t launch_step_advance(int32_t *step, int32_t n_steps, hipStream_t s) {
    hipLaunchKernelGGL(k_step_advance, dim3(1), dim3(64), 0, s, step, n_steps);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Streaming copy, 16 B per lane per step (n % 16 == 0).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, uint64_t n16) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

hipError_t launch_copy(const uint8_t *src, uint8_t *dst, uint64_t n, hipStream_t s) {
    const uint64_t n16 = n / 16;
    uint64_t grid = (n16 + 255) / 256;
    if (grid > 8192) grid = 8192;
    hipLaunchKernelGGL(k_copy, dim3((uint32_t)grid), dim3(256), 0, s, (const uint4 *)src, (uint4 *)dst, n16);
    return hipGetLastError();
}

}  // namespace kq
