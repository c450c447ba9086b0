// The non-fused AdamW step on 4-bit states with the reference's default scalings -- first
// moment block-wise over 128 values, second moment rank-1 (scale[r, c] = min(rowmax[r],
// colmax[c])) -- in two passes over HBM instead of the seven of the staged path
// (lpmm/optim/adamw.py:394-436: two dequantisations, the update, the statistics of the new
// second moment, two quantisations).
//
// The second moment cannot be re-quantised where it is computed, because its scales are
// maxima over whole rows and columns of the new values.  So:
//
//   pass 1 (update):   reads p, g, both code arrays and the current statistics; updates p,
//                      re-quantises m, and merges the row/column maxima of the new v into the
//                      next statistics (atomic max on the bit patterns: exact, order-free);
//   pass 2 (requant):  reads g, the old v codes and both sets of statistics, recomputes the
//                      new v with the same operations (bit-identical), normalises by the next
//                      statistics and overwrites the v codes in place.
//
// 18.5 bytes per parameter cross HBM instead of 50.  The column count must be a multiple of
// 128, so that the 128-value groups of m never straddle rows: 16 lanes (one DPP row) own 128
// consecutive columns of one tensor row.  A 256-thread workgroup covers tile_rows rows by
// 128 << lg_wide columns, per pass (16 >> lg_wide) rows of (1 << lg_wide) adjacent groups, so
// that its accesses to a row are contiguous runs of 512 << lg_wide bytes.
//
// Both kernels run at the rate the memory system gives to their access structure, not at that
// of their arithmetic (with the arithmetic taken out they take the same time).  Measured on the
// LLaMA-7B shapes: a workgroup that walks through many passes is slower than the same accesses
// made by short-lived workgroups in dispatch order (tiles of 1 or 2 passes run at the rate of
// the one-shot fused step, 8 passes over 16 rows by 1024 columns 13 % below it), but short
// tiles mean more column atomics and more tile set-up.  Tiles are 256 columns wide and 16 to 64 rows tall, by pass and
// by the size of the launch (pass_rows_policy).  The row blocks that are
// resident together interleave their passes (block k of a group of `comb` blocks takes the rows
// of pass i at (i * comb + k) * pass_rows), so that at any time a group works on one contiguous
// band of the tensor instead of on `comb` bands a tile apart.  Together 2130 -> 1990 us (first
// pass) and 770 -> 705 us (second pass) per launch of 8.4e8 elements.
#include "lpmm_plain.hpp"
#include "rank1_tiles.hpp"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace lpmm {

// Zeroes the arrays that the first pass merges maxima into: the next statistics, and the next scales of first-moment
// groups that are wider than 128 values or straddle rows.  Ranges of all tensors of a call in one launch (5 us each on an
// otherwise idle stream), neighbours in memory joined.  Two sizes of arguments: the host copies them whole.
constexpr int kClearMax = 480, kClearFew = 64;
template <int N>
struct ClearRanges {
    float *at[N];
    int64_t n[N];
};
static_assert(sizeof(ClearRanges<kClearMax>) <= kMostKernargBytes, "kernel arguments exceed 8 KB");

template <int N>
__device__ __forceinline__ void clear_range(const ClearRanges<N> &ranges, uint32_t range, uint32_t block, uint32_t blocks)
{
    float *const at = ranges.at[range];
    const int64_t n = ranges.n[range];
    for (int64_t i = (int64_t)block * kThreads + threadIdx.x; i < n; i += (int64_t)blocks * kThreads)
        at[i] = 0.0f;
}

template <int N>
__global__ __launch_bounds__(kThreads) void rank1_clear_kernel(const ClearRanges<N> ranges)
{
    clear_range(ranges, blockIdx.y, blockIdx.x, gridDim.x);
}

// The clearing, `blocks` workgroups a range, and tensors with fp32 states, whose own launch (4.7 us on the device, 4 to 5 on the host)
// this one saves: a step on one layer of width 64 34.2 -> 28.9 us, on two bottleneck blocks of width 64 40.7 -> 34.2, on 48 layers of width
// 448 (with one call for all their launches of 32 matrices) 473 -> 461.
constexpr int kClearJoined = 192;
template <int N>
__global__ __launch_bounds__(kThreads) void rank1_clear_plain_kernel(const ClearRanges<N> ranges, const MultiF plain, uint32_t blocks,
                                                                     uint32_t clears)
{
    if (blockIdx.x < clears)
        clear_range(ranges, blockIdx.x / blocks, blockIdx.x % blocks, blocks);
    else
        tile_fp32<NonFusedArith>(plain, blockIdx.x - clears);
}
static_assert(sizeof(ClearRanges<kClearJoined>) + sizeof(MultiF) + 8 <= kMostKernargBytes, "kernel arguments exceed 8 KB");
static_assert(kThreads == kPlainThreads, "tile_fp32 runs in these kernels");

// the first N of a call's ranges
template <int N>
static ClearRanges<N> ranges_from(const ClearRanges<kClearMax> &all)
{
    ClearRanges<N> r;
    memcpy(r.at, all.at, sizeof r.at);
    memcpy(r.n, all.n, sizeof r.n);
    return r;
}

static void launch_clear_plain(const ClearRanges<kClearMax> &ranges, int n, uint32_t blocks, PlainSet &plain, double beta1, double beta2,
                               double lr, double weight_decay, double eps, hipStream_t s)
{
    MultiF args;
    const NfHyper c = make_nf_hyper(beta1, beta2, lr, weight_decay, eps, 1.0);
    const float scalars[7] = {c.decay, c.w1, c.b2, c.w2, c.eps, 0.0f, 0.0f};
    memcpy(args.s, scalars, sizeof args.s);
    const int64_t first = plain.next;
    uint32_t tiles = fill_fp32(args, plain.tensors, plain.count, plain.next, [=](float step, float(&k)[4]) {
        NonFusedArith::per_tensor(beta1, beta2, lr, weight_decay, eps, step, k);
    });
    const uint32_t clears = (uint32_t)n * blocks;
    if (tiles > 0x7fffffffu - clears) {  // they go alone
        plain.next = first;
        tiles = 0;
    }
    if (n <= kClearFew)
        hipLaunchKernelGGL(rank1_clear_plain_kernel<kClearFew>, dim3(clears + tiles), dim3(kThreads), 0, s, ranges_from<kClearFew>(ranges),
                           args, blocks, clears);
    else
        hipLaunchKernelGGL(rank1_clear_plain_kernel<kClearJoined>, dim3(clears + tiles), dim3(kThreads), 0, s,
                           ranges_from<kClearJoined>(ranges), args, blocks, clears);
}

// What a kernel's tensors may be beside matrices of whole column blocks: double rows, which end with a whole row, or rows of several tensor
// rows, the last of which may be a part (rank1_tiles.hpp: Fold).
enum FoldKind : int { kNoFold = 0, kDoubles = 1, kWraps = 2 };

// operands of one pass of a DPP row, as loaded
struct PassRegs {
    float4 a0, a1, b0, b1;
    float4 c0, c1;  // fp32 first moment only
    uint32_t m0, m1, v0, v1;
    float sm, ro, ro1;  // ro1: the second tensor row's statistic (folded rows; otherwise ro)
};

template <int MODE, int FOLD, bool KEEP>
__device__ __forceinline__ void pass_fetch(const TensorR1 &t, const Fold &f, const FoldSpan &span, uint32_t cg, int lane16, int64_t r,
                                           PassRegs &x)
{
    const int64_t grp = r * f.col_blocks + cg;
    const int64_t gbase = grp * kGroup;
    if (FOLD == kWraps) {
        // runs beyond the end read the last one
        const int64_t last = f.values - 4, oa = gbase + lane16 * 4, ob = oa + 64;
        const int64_t a = oa < last ? oa : last, b = ob < last ? ob : last;
        x.a0 = load4(t.p + a);
        x.a1 = load4(t.p + b);
        x.b0 = load4_for<KEEP>(t.g + a);
        x.b1 = load4_for<KEEP>(t.g + b);
        if (MODE == kMFloat) {
            x.c0 = load4(reinterpret_cast<const float *>(t.mc) + a);
            x.c1 = load4(reinterpret_cast<const float *>(t.mc) + b);
        } else {
            x.m0 = load_u16(reinterpret_cast<const uint16_t *>(t.mc + (a >> 1)));
            x.m1 = load_u16(reinterpret_cast<const uint16_t *>(t.mc + (b >> 1)));
            x.sm = t.ms[MODE == kMCodesWide ? (a >> 7) >> t.m_lg : a >> 7];
        }
        x.v0 = load_u16_for<KEEP>(reinterpret_cast<const uint16_t *>(t.vc + (a >> 1)));
        x.v1 = load_u16_for<KEEP>(reinterpret_cast<const uint16_t *>(t.vc + (b >> 1)));
        int64_t r0, r1;
        fold_rows(f, span, r, r0, r1);
        x.ro = t.row_old[r0];
        x.ro1 = t.row_old[r1];
        return;
    }
    const float *pp = t.p + gbase + lane16 * 4;
    const float *gp = t.g + gbase + lane16 * 4;
    x.a0 = load4(pp);
    x.a1 = load4(pp + 64);
    x.b0 = load4_for<KEEP>(gp);
    x.b1 = load4_for<KEEP>(gp + 64);
    const uint16_t *vcp = reinterpret_cast<const uint16_t *>(t.vc + (gbase >> 1)) + lane16;
    if (MODE == kMFloat) {
        const float *mp = reinterpret_cast<const float *>(t.mc) + gbase + lane16 * 4;
        x.c0 = load4(mp);
        x.c1 = load4(mp + 64);
    } else {
        const uint16_t *mcp = reinterpret_cast<const uint16_t *>(t.mc + (gbase >> 1)) + lane16;
        x.m0 = load_u16(mcp);
        x.m1 = load_u16(mcp + 16);
        x.sm = t.ms[MODE == kMCodesWide ? grp >> t.m_lg : grp];
    }
    x.v0 = load_u16_for<KEEP>(vcp);
    x.v1 = load_u16_for<KEEP>(vcp + 16);
    if (FOLD) {
        uint32_t halves[2];
        double_halves(f, cg, halves);
        x.ro = t.row_old[(r << f.lg) + halves[0]];
        x.ro1 = t.row_old[(r << f.lg) + halves[1]];
    } else {
        x.ro = x.ro1 = t.row_old[r];
    }
}

#ifndef LPMM_R1_WAVES
#define LPMM_R1_WAVES 4
#endif
// 4 waves per SIMD, up to 128 registers: the first pass's operands stay live across the prologue and
// the lane's column statistics across the passes (with 5 or 6 the compiler spills or re-reads)
template <int MODE, int FOLD, bool KEEP, int N>
__global__ __launch_bounds__(kThreads, LPMM_R1_WAVES) void rank1_update_kernel(const MultiR1N<N> args, const float *__restrict__ qmap_m,
                                                                const float *__restrict__ qmap_v)
{
    constexpr int kSlots = FOLD == kWraps ? kFoldSlots : kRowSlots;
    static_assert(FOLD != kDoubles || MODE == kMCodes128, "double rows: 4-bit first moments in groups of 128 values");
    __shared__ __align__(16) uint32_t lds[(kColExtra + kMaxWide * kRedSlotWords * 4) / 4 + kSlots];
    uint32_t *colred = lds + kColExtra / 4;
    uint32_t *rowred = colred + kMaxWide * kRedSlotWords;
    const int lo = find_tensor(args);
    const TensorR1 &t = args.t[lo];
    const uint32_t tl = blockIdx.x - args.tile_start[lo];
    const int lane16 = threadIdx.x & 15, drow = threadIdx.x >> 4;
    const Fold f = fold_of<FOLD != kNoFold>(t);
    const Geometry q = geometry(t.tile, f.col_blocks, tl, drow);
    const int64_t cols = (int64_t)f.col_blocks * kGroup;
    const int64_t tile_c0 = (int64_t)q.col_tile * q.wide * kGroup;

    // Order of the prologue: the small loads that feed LDS (maps, encode table, the tile's current
    // column statistics), then the streaming loads of the first pass, then the LDS writes (the
    // small loads were issued first and return first) and a barrier that orders LDS only -- the
    // first pass's operands are on their way while the tables are set up.
    const LdsFill fill = lds_fill_load(qmap_m, qmap_v);
    constexpr int kColPerThread = kMaxWide * kGroup / kThreads;
    uint32_t co_in[kColPerThread];
#pragma unroll
    for (int i = 0; i < kColPerThread; ++i) {
        const int j = threadIdx.x + i * kThreads;
        co_in[i] = (j < q.wide * kGroup && tile_c0 + j < cols)
                       ? __float_as_uint(t.col_old[FOLD ? fold_col(f, (uint32_t)(tile_c0 + j)) : tile_c0 + j])
                       : 0u;
    }
    const bool row_live = q.cg < f.col_blocks;  // the whole DPP row
    // No branch around the first pass's loads: behind one the compiler waits for all of them before the LDS writes, as the path without
    // them has nothing else to count.  A DPP row without work loads what is there.
    PassRegs x;
    const uint32_t cg = row_live ? q.cg : f.col_blocks - 1u;
    const FoldSpan span = FOLD == kWraps ? fold_span(f, cg) : FoldSpan{0, kGroup};
    pass_fetch<MODE, FOLD, KEEP>(t, f, span, cg, lane16, q.row0 < f.rows ? q.row0 : f.rows - 1, x);
    lds_fill_store(lds, fill);
    for (int j = threadIdx.x; j < kMaxWide * (int)kRedSlotWords; j += kThreads)
        colred[j] = 0u;
    for (int j = threadIdx.x; j < kSlots; j += kThreads)
        rowred[j] = 0u;
#pragma unroll
    for (int i = 0; i < kColPerThread; ++i)
        lds[kColOld / 4 + threadIdx.x + i * kThreads] = co_in[i];
    const int kind_m = classify_map(qmap_m);
    NfHyper h;
    h.decay = args.decay;
    h.w1 = args.w1;
    h.b2 = args.b2;
    h.w2 = args.w2;
    h.eps = args.eps;
    h.neg_step_size = t.neg_step_size;
    h.bc2_sqrt = t.bc2_sqrt;
    h.rbc2_sqrt = t.rbc2_sqrt;
    lds_barrier();

    if (MODE == kMCodes128 && tl == 0) {
        const float z[kEltsPerLane] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        const int64_t n = (f.values + kGroup - 1) / kGroup * kGroup;
        write_padding(t.mc, n, (n + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP,
                      encode8_plain(lds, kLdsQ0, kind_m, z));
    }

    const int slot = drow & (q.wide - 1);
    if (row_live) {
        const uint32_t co_off = kColOld + (slot * kGroup + lane16 * 4) * 4;
        uint32_t *red = colred + slot * kRedSlotWords + lane16;
        // folded rows: do the lane's two runs take the second of the two row statistics
        const bool second_a = FOLD == kWraps && (uint32_t)(4 * lane16) >= span.split;
        const bool second_b = FOLD == kDoubles || (FOLD == kWraps && (uint32_t)(64 + 4 * lane16) >= span.split);
        const uint32_t in_tile = FOLD != kWraps ? 0u : span.first - fold_span(f, q.col_tile * (uint32_t)q.wide).first;
        // a lane keeps its eight columns through all passes: their statistics come out of LDS once
        float co[kEltsPerLane];
        unpack8(lds_read<float4>(lds, co_off), lds_read<float4>(lds, co_off + 256), co);
        const float least = t.tile.drop_nan ? 0.0f : __builtin_nanf("");  // of a column's values
#pragma unroll 1
        for (int it = 0; it < q.passes; ++it) {
            const int64_t r = q.row0 + it * q.step;
            const int64_t grp = r * f.col_blocks + q.cg;
            const int64_t gbase = grp * kGroup;
            if (r >= f.rows || (FOLD == kWraps && gbase >= f.values))
                break;
            if (it > 0)
                pass_fetch<MODE, FOLD, KEEP>(t, f, span, q.cg, lane16, r, x);
            const bool live_a = FOLD != kWraps || gbase + 4 * lane16 < f.values, live_b = FOLD != kWraps || gbase + 4 * lane16 + 64 < f.values;
            float *pp = t.p + gbase + lane16 * 4;
            const uint32_t wv = x.v0 | (x.v1 << 16);
            const float ro_a = second_a ? x.ro1 : x.ro, ro_b = second_b ? x.ro1 : x.ro;
            float pv[kEltsPerLane], gv[kEltsPerLane], m[kEltsPerLane], v[kEltsPerLane];
            unpack8(x.a0, x.a1, pv);
            unpack8(x.b0, x.b1, gv);
            constexpr bool M32 = MODE == kMFloat;
            const Nibbles nm = split_nibbles(M32 ? 0u : (x.m0 | (x.m1 << 16)));
            const float sm = M32 ? 0.0f : x.sm;
            if (M32)
                unpack8(x.c0, x.c1, m);

            const Nibbles nv = split_nibbles(wv);
            float amax_m = 0.0f, vmax = 0.0f, vmax1 = 0.0f;  // vmax1: the second tensor row's (folded rows)
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                if (!M32)
                    m[k] = decode_nibble(lds, kLdsQ0, nm, k) * sm;
                const float rk = k >= 4 ? ro_b : ro_a;
                v[k] = decode_nibble(lds, kLdsQ1, nv, k) * ((co[k] < rk) ? co[k] : rk);
            }
            if (FOLD == kWraps && !live_b) {
                // beyond the end: the zeros that fill up the last group
#pragma unroll
                for (int k = 0; k < kEltsPerLane; ++k)
                    if (k >= 4 || !live_a)
                        gv[k] = m[k] = v[k] = 0.0f;
            }
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                nonfused_elt(pv[k], gv[k], m[k], v[k], h);
                amax_m = fmaxf(amax_m, fabsf(m[k]));
                if (FOLD && k >= 4)
                    vmax1 = fmaxf(vmax1, v[k]);
                else
                    vmax = fmaxf(vmax, v[k]);
                atomicMax(red + k * 16, __float_as_uint(FOLD == kWraps ? fmaxf(v[k], least) : v[k]));
            }
            if (FOLD == kWraps) {
                const float a = vmax, b = vmax1;
                vmax = fmaxf(second_a ? 0.0f : a, second_b ? 0.0f : b);
                vmax1 = fmaxf(second_a ? a : 0.0f, second_b ? b : 0.0f);
            }
            uint32_t cm = 0;
            if (M32) {
                vmax = row16_max(vmax);
            } else {
                row16_max2(amax_m, vmax);
                if (MODE == kMCodes128)
                    cm = encode8_scaled(lds, kLdsQ0, kind_m, m, amax_m);
            }
            if (FOLD)
                vmax1 = row16_max(vmax1);

            if (live_a)
                store4(pp, make_float4(pv[0], pv[1], pv[2], pv[3]));
            if (live_b)
                store4(pp + 64, make_float4(pv[4], pv[5], pv[6], pv[7]));
            if (M32) {
                float *mp = reinterpret_cast<float *>(t.mc) + gbase + lane16 * 4;
                if (live_a)
                    store4(mp, make_float4(m[0], m[1], m[2], m[3]));
                if (live_b)
                    store4(mp + 64, make_float4(m[4], m[5], m[6], m[7]));
            } else if (MODE == kMCodes128) {
                uint16_t *mcp = reinterpret_cast<uint16_t *>(t.mc + (gbase >> 1)) + lane16;
                store_u16(mcp, cm & 0xFFFFu);
                store_u16(mcp + 16, cm >> 16);
                if (lane16 == 0)
                    t.ms[grp] = amax_m;
            } else if (lane16 == 0) {
                atomic_max_nonneg(t.ms_new + (grp >> t.m_lg), amax_m);
            }
            if (lane16 == 0) {
                // the maxima of a tensor row meet in LDS (rank1_tiles.hpp)
                uint32_t *slot = rowred + row_slot(t.tile, it, drow) * (FOLD == kWraps ? 2 : 1);
                if (FOLD == kDoubles) {
                    uint32_t halves[2];
                    double_halves(f, q.cg, halves);
                    atomicMax(slot + halves[0], __float_as_uint(vmax));
                    atomicMax(slot + halves[1], __float_as_uint(vmax1));
                } else if (FOLD) {
                    atomicMax(slot + in_tile, __float_as_uint(vmax));
                    if (span.split < (uint32_t)kGroup)
                        atomicMax(slot + in_tile + 1, __float_as_uint(vmax1));
                } else {
                    atomicMax(slot, __float_as_uint(vmax));
                }
            }
        }
    }
    // the column maxima meet in LDS: nothing below depends on the global stores still in flight
    lds_barrier();
    if (FOLD == kWraps)
        flush_row_maxima_fold(rowred, t.tile, q, drow, f, t.row_new);
    else
        flush_row_maxima(rowred, t.tile, q, drow, f.rows, t.row_new, f.lg);
    // column j of the tile = element k of lane l of slot s
    for (int j = threadIdx.x; j < q.wide * kGroup; j += kThreads) {
        const int w = j & (kGroup - 1);
        const int k = ((w >> 6) << 2) | (w & 3), l = (w >> 2) & 15;
        if (tile_c0 + j < cols) {
            float *dst = t.col_new + (FOLD ? fold_col(f, (uint32_t)(tile_c0 + j)) : tile_c0 + j);
            const uint32_t mine = colred[(j >> 7) * kRedSlotWords + k * 16 + l];
            atomic_max_nonneg(dst, __uint_as_float(mine));
        }
    }
}

// The runs of a lane beyond the end of the tensor: the second, and the first with it.
__device__ __forceinline__ void zero_beyond(float (&x)[kEltsPerLane], bool both)
{
#pragma unroll
    for (int k = 0; k < kEltsPerLane; ++k)
        if (k >= 4 || both)
            x[k] = 0.0f;
}

// MWIDE: the first moment's groups are wider than 128 values; its codes are written here too.
template <bool MWIDE, int FOLD, int N>
__global__ __launch_bounds__(kThreads) void rank1_requant_kernel(const MultiR1N<N> args, const float *__restrict__ qmap_m,
                                                                 const float *__restrict__ qmap_v)
{
    __shared__ __align__(16) uint32_t lds[(kColExtra + 2 * kColBytes) / 4];
    constexpr uint32_t kColNew = kColExtra, kColRcp = kColExtra + kColBytes;
    constexpr uint32_t kVMap = MWIDE ? kLdsQ1 : kLdsQ0;  // where the second moment's map sits in LDS
    if (MWIDE)
        lds_fill(lds, qmap_m, qmap_v);
    else
        lds_fill(lds, qmap_v, nullptr);
    const int kind = classify_map(qmap_v);
    const int kind_m = MWIDE ? classify_map(qmap_m) : kMapGeneric;
    const int lo = find_tensor(args);
    const TensorR1 &t = args.t[lo];
    const uint32_t tl = blockIdx.x - args.tile_start[lo];
    const int lane16 = threadIdx.x & 15, drow = threadIdx.x >> 4;
    const Fold f = fold_of<FOLD != kNoFold>(t);
    const Geometry q = geometry(t.tile, f.col_blocks, tl, drow);
    const int64_t cols = (int64_t)f.col_blocks * kGroup;
    const int64_t tile_c0 = (int64_t)q.col_tile * q.wide * kGroup;
    for (int j = threadIdx.x; j < q.wide * kGroup; j += kThreads) {
        const bool in = tile_c0 + j < cols;
        const int64_t c = FOLD ? fold_col(f, (uint32_t)(tile_c0 + j)) : tile_c0 + j;
        const float cn = in ? t.col_new[c] : 0.0f;
        lds[kColOld / 4 + j] = in ? __float_as_uint(t.col_old[c]) : 0u;
        lds[kColNew / 4 + j] = __float_as_uint(cn);
        lds[kColRcp / 4 + j] = __float_as_uint(1.0f / cn);
    }
    NfHyper h;
    h.b2 = args.b2;
    h.w2 = args.w2;
    h.w1 = args.w1;
    __syncthreads();

    if (tl == 0) {
        const float z[kEltsPerLane] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        const int64_t n = FOLD ? (f.values + kGroup - 1) / kGroup * kGroup : f.values;
        const int64_t n_pack = (n + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP;
        write_padding(t.vc, n, n_pack, encode8_plain(lds, kVMap, kind, z));
        if (MWIDE) {
            // The quantiser pads the flattened tensor with zeros to whole groups (functional.py:404-422),
            // the packing pads to whole pack groups of 2048 values.  The zeros that fill up the last
            // group are divided by its scale like its other values (0/0 -> NaN -> code 15 when the
            // group is all zero), those behind it are plain zeros.
            const int64_t group = (int64_t)kGroup << t.m_lg;
            const int64_t n_grp = (n + group - 1) / group * group;
            const int64_t n_all = (n_grp + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP;
            const uint32_t zero_word = encode8_plain(lds, kLdsQ0, kind_m, z);
            uint32_t last_word = zero_word;
            if (n_grp > n) {
                const float last = t.ms_new[(n - 1) >> (7 + t.m_lg)];
                const float zs[kEltsPerLane] = {0.0f / last, 0.0f / last, 0.0f / last, 0.0f / last,
                                                0.0f / last, 0.0f / last, 0.0f / last, 0.0f / last};
                last_word = encode8_plain(lds, kLdsQ0, kind_m, zs);
            }
            for (int64_t i = n + (int64_t)threadIdx.x * kEltsPerLane; i < n_all; i += kThreads * kEltsPerLane)
                *reinterpret_cast<uint32_t *>(t.mc + (i >> 1)) = i < n_grp ? last_word : zero_word;
            if (threadIdx.x == 0)
                t.mc[n_all / 2] = 0;
        }
    }
    if (q.cg >= f.col_blocks)
        return;

    // a lane keeps its eight columns through all passes: their old and new statistics and the
    // reciprocals of the new ones come out of LDS once
    const uint32_t col_off = ((drow & (q.wide - 1)) * kGroup + lane16 * 4) * 4;
    float co[kEltsPerLane], cn[kEltsPerLane], rcn[kEltsPerLane];
    unpack8(lds_read<float4>(lds, kColOld + col_off), lds_read<float4>(lds, kColOld + col_off + 256), co);
    unpack8(lds_read<float4>(lds, kColNew + col_off), lds_read<float4>(lds, kColNew + col_off + 256), cn);
    unpack8(lds_read<float4>(lds, kColRcp + col_off), lds_read<float4>(lds, kColRcp + col_off + 256), rcn);
    bool cols_safe = true;
#pragma unroll
    for (int k = 0; k < kEltsPerLane; ++k)
        cols_safe = cols_safe && rc_safe(cn[k]) && co[k] == co[k];
    // the group's 64 code bytes move as one dword per lane (whole lines per access; with the
    // arithmetic taken out this pass is 11 % faster than with two 16-bit accesses per lane)
    const uint32_t code_dword = code_dword_of_lane(lane16), code_sel = code_swap_selector(lane16);
    const FoldSpan span = FOLD == kWraps ? fold_span(f, q.cg) : FoldSpan{0, kGroup};
    uint32_t halves[2] = {0u, 0u};
    if (FOLD == kDoubles)
        double_halves(f, q.cg, halves);
    // folded rows: do the lane's two runs take the second of the two row statistics
    const bool second_a = FOLD == kWraps && (uint32_t)(4 * lane16) >= span.split;
    const bool second_b = FOLD == kDoubles || (FOLD == kWraps && (uint32_t)(64 + 4 * lane16) >= span.split);
    const float most = FOLD == kWraps && t.tile.drop_nan ? 1.0f : __builtin_nanf("");
#pragma unroll 1
    for (int it = 0; it < q.passes; ++it) {
        const int64_t r = q.row0 + it * q.step;
        const int64_t gbase = (r * f.col_blocks + q.cg) * kGroup;
        if (r >= f.rows || (FOLD == kWraps && gbase >= f.values))
            break;
        const int64_t oa = gbase + lane16 * 4, ob = oa + 64, last = f.values - 4;
        int64_t r0 = r, r1 = r;  // the tensor rows of the DPP row
        if (FOLD == kWraps) {
            fold_rows(f, span, r, r0, r1);
        } else if (FOLD) {
            r0 = (r << f.lg) + halves[0];
            r1 = (r << f.lg) + halves[1];
        }
        // runs beyond the end read the last one
        const float4 b0 = load4(t.g + (FOLD == kWraps && oa > last ? last : oa)), b1 = load4(t.g + (FOLD == kWraps && ob > last ? last : ob));
        uint32_t *vcp = reinterpret_cast<uint32_t *>(t.vc + (gbase >> 1)) + code_dword;
        const uint32_t in_v = load_u32(vcp);
        const float ro = t.row_old[r0], rn = t.row_new[r0];
        const float ro1 = FOLD ? t.row_old[r1] : ro, rn1 = FOLD ? t.row_new[r1] : rn;
        uint32_t *mcp = nullptr;
        uint32_t wm = 0;
        float ms_old = 0.0f, ms_new = 0.0f;
        if (MWIDE) {
            mcp = reinterpret_cast<uint32_t *>(t.mc + (gbase >> 1)) + code_dword;
            const uint32_t in_m = load_u32(mcp);
            const int64_t mg = gbase >> (7 + t.m_lg);
            ms_old = t.ms[mg];
            ms_new = t.ms_new[mg];
            wm = swap_code_halves(in_m, code_sel);
        }
        const uint32_t wv = swap_code_halves(in_v, code_sel);
        float gv[kEltsPerLane], v[kEltsPerLane], x[kEltsPerLane];
        unpack8(b0, b1, gv);
        const Nibbles nv = split_nibbles(wv);
        // Every statistic the wave touches is a number, and the new ones lie in the range in which the
        // reciprocal is exact?  Then minima and maxima of these non-negative values can be taken on their
        // bit patterns (one instruction each), and the reciprocal of the smaller statistic is the larger
        // of the two reciprocals (rounding is monotonic).
        // (Where that saves registers as well -- double rows, wide first-moment groups -- it is 0.4-3 %
        // of the step; the plain variant would go from 74 to 82 registers and lose a wave per SIMD.)
        constexpr bool kBitMin = FOLD || MWIDE;
        const bool fast = kind == kMapStdV && __all(cols_safe && rc_safe(rn) && rc_safe(rn1) && ro == ro && ro1 == ro1);
        const float ro_a = second_a ? ro1 : ro, ro_b = second_b ? ro1 : ro, rn_a = second_a ? rn1 : rn, rn_b = second_b ? rn1 : rn;
        if (kBitMin && fast) {
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                const float rk = k >= 4 ? ro_b : ro_a;
                v[k] = decode_nibble(lds, kVMap, nv, k) * __uint_as_float(min(__float_as_uint(co[k]), __float_as_uint(rk)));
                nonfused_second_moment(v[k], gv[k], h);
            }
        } else {
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                const float rk = k >= 4 ? ro_b : ro_a;
                v[k] = decode_nibble(lds, kVMap, nv, k) * ((co[k] < rk) ? co[k] : rk);
                nonfused_second_moment(v[k], gv[k], h);
            }
        }
        if (MWIDE) {
            // the first moment as the update pass computed it, with the scale of its whole group
            const Nibbles nm = split_nibbles(wm);
            float m[kEltsPerLane];
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k)
                m[k] = lerp_w(decode_nibble(lds, kLdsQ0, nm, k) * ms_old, gv[k], h.w1);
            if (FOLD == kWraps && ob > last)
                zero_beyond(m, oa > last);
            store_u32(mcp, swap_code_halves(encode8_scaled(lds, kLdsQ0, kind_m, m, ms_new), code_sel));
        }
        uint32_t w;
        // every scale the wave divides by is a column or the row statistic: all in the range in
        // which the reciprocal is exact?
        if (fast) {
            // the correctly rounded reciprocal of whichever statistic is the scale, then one
            // multiply and two fmas: the correctly rounded quotient (v <= scale by construction)
            const float rcr = rcp_exact(rn_a), rcr1 = FOLD ? rcp_exact(rn_b) : rcr;
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                const float rnk = k >= 4 ? rn_b : rn_a, rck = (FOLD && k >= 4) ? rcr1 : rcr;
                if (kBitMin) {
                    const float sk = __uint_as_float(min(__float_as_uint(cn[k]), __float_as_uint(rnk)));
                    const float rk = __uint_as_float(max(__float_as_uint(rcn[k]), __float_as_uint(rck)));
                    x[k] = div_by_rc(v[k], sk, rk);
                } else {
                    const bool by_col = cn[k] < rnk;
                    x[k] = div_by_rc(v[k], by_col ? cn[k] : rnk, by_col ? rcn[k] : rck);
                }
            }
            if (FOLD == kWraps) {
                // a NaN whose column's statistic leaves it out: code 15
#pragma unroll
                for (int k = 0; k < kEltsPerLane; ++k)
                    x[k] = fminf(x[k], most);
                if (ob > last)
                    zero_beyond(x, oa > last);
            }
            w = encode8_std_v(x);
        } else {
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                const float rnk = k >= 4 ? rn_b : rn_a;
                x[k] = v[k] / ((cn[k] < rnk) ? cn[k] : rnk);
            }
            if (FOLD == kWraps && ob > last)
                zero_beyond(x, oa > last);
            w = encode8_plain(lds, kVMap, kind, x);
        }
        store_u32(vcp, swap_code_halves(w, code_sel));
    }
}

}  // namespace lpmm

using namespace lpmm;

// The widest tile the policy allows (longest contiguous runs) that leaves at most 10 % of the DPP
// rows of a tensor's tiles without a column group; otherwise the width that wastes least.  (13
// column groups, 1600 columns: tiles of two groups with one DPP row in 14 idle run 4 % faster than
// tiles of one group.)
static uint32_t choose_lg_wide(uint32_t col_blocks)
{
    uint32_t best = 0;
    double best_use = 0.0;
    for (int lg = kPolicyLgWide; lg >= 0; --lg) {
        const uint32_t wide = 1u << lg;
        const double use = (double)col_blocks / (double)((col_blocks + wide - 1) / wide * wide);
        if (use >= 0.90)
            return (uint32_t)lg;
        if (use > best_use) {
            best_use = use;
            best = (uint32_t)lg;
        }
    }
    return best;
}

constexpr double kValuesPerRowBlock = 12000;  // pass_rows_policy
constexpr uint64_t kCombMultiple = 8;
static_assert(kPolicyResident % kCombMultiple == 0, "a rounded group is no larger than the resident set");

// Row blocks of a matrix, and its tiles side by side.
struct Blocks {
    uint32_t lg_wide, tile_rows;
    uint64_t rows, col_tiles;
};

static Blocks blocks_of(int64_t rows, uint32_t col_blocks, uint32_t policy_rows)
{
    Blocks b;
    b.lg_wide = choose_lg_wide(col_blocks);
    b.col_tiles = (col_blocks + (1u << b.lg_wide) - 1) >> b.lg_wide;
    const uint32_t pass_rows = (uint32_t)kDppRows >> b.lg_wide;
    b.tile_rows = pass_rows > policy_rows ? pass_rows : policy_rows;
    b.rows = (uint64_t)((rows + b.tile_rows - 1) / b.tile_rows);
    return b;
}

// Tile shape of a rows x (128 * col_blocks) tensor, and its tile count.  Row blocks interleave in groups of as many as are resident
// together.
// spread: what is left for the last group goes to as many blocks, each with fewer passes.  In launches of few workgroups these
// short ones even out what the CUs have to do (LaunchKind::spread).
static uint64_t shape_tiles(int64_t rows, uint32_t col_blocks, TileShape &ts, uint32_t policy_rows, bool spread)
{
    const Blocks b = blocks_of(rows, col_blocks, policy_rows);
    uint64_t comb = kPolicyResident / b.col_tiles;
    comb = comb < 1 ? 1 : comb;
    if (spread) {
        comb = comb > b.rows ? b.rows : comb;
    } else {
        // groups of equal size, so that the last one holds few empty blocks (13 row blocks in groups of 5, not 6)
        const uint64_t groups = (b.rows + comb - 1) / comb;
        comb = (b.rows + groups - 1) / groups;
        // Large groups (narrow matrices) hold a multiple of 8 blocks: neighbours share cache lines of row statistics and scales, and with
        // an odd number the sharing blocks, and the XCDs they are on, change from pass to pass.  Update and second pass, equal groups ->
        // multiples of 8: 50257 x 128 31.7 / 10.9 -> 29.1 / 9.1 us, 100000 x 128 49.2 / 16.0 -> 49.3 / 14.9.  (Multiples of 32 leave more
        // blocks empty: a step on 24 of 12592 x 278 632 -> 660.)
        if (comb >= 64)
            comb = (comb + kCombMultiple - 1) / kCombMultiple * kCombMultiple;
    }
    ts.lg_wide = b.lg_wide;
    ts.drop_nan = 0;
    ts.tile_rows = b.tile_rows;
    ts.comb = (uint32_t)comb;
    return (b.rows + comb - 1) / comb * comb * b.col_tiles;
}

// The matrix that a pass's tiles cover; can_fold: column counts that are no multiple of 128 are folded (and satisfy can_fold_rows).
struct Matrix {
    int64_t rows;
    uint32_t col_blocks, lg;
};

static Matrix matrix_of(int64_t rows, int64_t cols, bool can_fold)
{
    if (!can_fold || cols % kGroup == 0)
        return {rows, (uint32_t)((cols + kGroup - 1) / kGroup), 0};
    const uint32_t lg = fold_lg((uint32_t)cols);
    return {(rows + ((int64_t)1 << lg) - 1) >> lg, (uint32_t)(cols >> (7 - lg)), lg};
}

// What a launch is, as far as its tile shapes depend on it.
struct LaunchKind {
    bool half_io, m32, bits;
    double values;  // of all its tensors
    bool spread[2];  // update pass, second pass: see shape_tiles
};

// Launches of fewer workgroups than are resident together have their remainders spread: those of the float16 kernels and of the
// ones for any column count, whose tiles take longest, and those of one tensor.  Update and second pass (us; equal groups ->
// spread): float16 6974 x 3840 59.6 / 24.8 -> 53.2 / 23.5, 1962 x 6831 61.8 / 89.3 -> 54.7 / 84.2, 39877 x 128 27.7 / 10.7 ->
// 24.1 / 9.2, but a step on four of 39394 x 128 (1232 workgroups) 74 -> 78, 11008 x 4096 (1376) 84.1 / 34.1 -> 86.0 / 35.6, eight
// of 962 x 9856 (2496) 141.5 / 60.0 -> 155.6 / 63.5; second pass on 1071 x 7515 51.4 -> 45.9, at 8 bits 28.8 -> 24.0; float32
// 21788 x 256 24.9 / 7.9 -> 23.4 / 7.3, 20000 x 128 15.8 / 5.4 -> 15.0 / 5.5, but four of 482 x 4608 26 / 10.4 -> 26 / 12.2.
constexpr uint64_t kSpreadBelow = 1024;

// Rows of a pass's tiles on a matrix of `rows` rows.  A tile of fewer rows means more column atomics and more set-up, one of
// more rows a longer walk, fewer workgroups and a longer end of the launch.  Measured (us; update pass, then second pass):
//   * few values leave the chip idle with tall tiles.  2048 x 2048 alone: 64 rows 22.3 / 10.0, 32 rows 15.9 / 7.9, 16 rows
//     14.2 / 7.3; 32 weights of 256 x 2304: 59 / 21, 52 / 22, 50 / 24; of 512 x 2048: 90 / 37, 87 / 35, 84 / 43; 24 of
//     1600 x 6400 (246M values): 571 / 209, 560 / 218, 578 / 274.  So the second pass goes below 64 rows only under
//     14M values, the update pass under 64M;
//   * tiles of one column group (narrow matrices, odd numbers of groups) hold half as many values, so their limits lie at fewer.
//     24 of 3760 x 128: 16 rows 40.7 / 18.4, 32 rows 32.3 / 14.7, 64 rows 31.6 / 12.5; 8 of 4000 x 384: 43.3 / 21.5, 34.4 / 15.8, 34.8 /
//     12.4; 8 of 9000 x 128: 44.5 / 14.8, 31.0 / 12.1, 27.0 / 9.9; second pass on 5000 x 640 8.2, 6.7, 7.5, on 4000 x 640 16 rows 6.3,
//     32 rows 6.8; but 24 of 600 x 128 8.2 / 5.7, 8.7 / 6.0, 12.4 / 6.8;
//   * byte codes gain less from short tiles: update of 4096 x 4096 56 with 16 rows, 51.6 with 32, 50.4 with 64, of 24 of 4000 x 256 85.0,
//     74.3, 79.2, of 8 of 626 x 2304 (11.5M values) 39.3, 40.3, 39.8, of 6 of 2000 x 640 31.5, 28.2, 26.6;
//   * no more than 256 row blocks of 16 rows on a column: their atomics on one address queue up (8192 x 256 among 5.5M
//     values: 16 rows 27.2, 32 rows 20.9), nor many more than 256 of 32 rows (21788 x 256: 32 rows 42.5, 64 rows 36.0 to 38.8);
//   * larger launches: the update pass does best with 32 rows where a DPP row is a whole column block (LLaMA-7B decoder
//     layers 1853 -> 1818), with 16 where the first moment is fp32 (a pass moves 20.5 instead of 13.5 bytes a value; a step of
//     these layers with 64, 32, 24, 16 rows: 3515, 3425, 3375, 3333) and with 64 where rows fold (GPT-2-XL's set 5590 ->
//     5549 a step); for byte codes 32 and 64 rows are the same (2925, 2916 a step, within the spread of one side's runs).
//   * whatever the launch holds, a column takes no more row blocks than one per 12000 values of its matrix, or 512: 18 ns an atomic on
//     one address are then less than the time of its values (13.5 to 20.5 bytes each at 6 TB/s).  Steps with tiles of 16, 32, 64, 128
//     rows: 1048576 x 128 1377, 777, 498, 450 (fp32 first moment 1379, 805, 628, 621; 8 bits 1406, 822, 508, 504), 524288 x 256
//     769, 492, 448, 443, 262144 x 512 492, 426, 430, 438, 131072 x 1024 419, 421, 428, 437 (fp32 573, 584, 596, 605);
//   * rows of an odd column count: the second pass sets the 4-bit codes of shared bytes by atomics, which shorter tiles spread.  Six
//     tensors of 4095 x 4099: 64 rows 657, 32 rows 630, 16 rows 614 (fp32 first moment 414, 396, 376); 5000 x 5001 128, 127, 123; 2072 x 4615
//     50, 59 (1235 workgroups, a fifth more than are resident together), 52; ten of 1001 x 1003 54, 58, 51; but 2001 x 3001 40, 34, 36.
// The float16 update is bound by its arithmetic, so that large launches take tall tiles, which spread a tile's set-up; small ones
// leave the chip idle with them.  Update / second pass with tiles of 128, 64, 32, 16 rows: 20 of 4096 x 11008 (902M values) 1323 / 495, 1333 /
// 518, 1391 / 509, 1507 / 743; 8 of 4096 x 4096 233 / 91, 225 / 90; 4 of them 102 / 47, 97 / 42, 103 / 43 (so that up to
// some 200M values 64 rows would take 3 to 7 % less; from 26M on the rows are 128 all the same, with which the groups of kSpreadBelow were
// measured: 6974 x 3840); one 35.8 / 18.7, 31.1 / 14.0,
// 30.2 / 14.6, 32.6 / 16.4; 24 of 512 x 2048 45.8 / 21.9, 41.5 / 18.3, 42.7 / 19.5; 32 of 256 x 2304 43.6 / 20.7, 35.8 / 15.9, 33.6 / 16.2,
// 36.6 / 18.4; 8 of 1024 x 1024 28.7 / 16.4, 21.0 / 11.0, 19.0 / 8.9, 19.6 / 10.2; 24 of 512 x 512 27.9 / 15.5, 20.5 / 11.0, 16.5 /
// 8.3, 15.7 / 7.9; update of 39877 x 128 22.6, 29.0 (a column's row blocks).  Any column count likewise: 2001 x 3001 49.5 / 82, 29.7, 30.2, 30.3 / 35.8;
// 6 of 4096 x 4100 297, 288, 292, 306.
static uint32_t pass_rows_policy(const LaunchKind &l, bool requant, const Matrix &m, bool odd_cols)
{
    const bool fold = m.lg != 0;
    const uint32_t col_blocks = m.col_blocks;
    const double values = (double)m.rows * (double)col_blocks * kGroup;
    // a row block has as many atomics on a column as the fold has rows; double rows count as one
    const int64_t rows = fold ? m.rows << (m.lg - 1) : m.rows;
    if (l.half_io && requant)
        return l.values < 6.5e6 ? kPolicyRows / 4 : l.values < 14e6 ? kPolicyRows / 2 : l.values < 26e6 ? kPolicyRows : kPolicyRowsHalf;
    const bool single = choose_lg_wide(col_blocks) == 0;  // tiles of one column group
    if (requant && odd_cols && !l.bits)
        return l.values >= (single ? 3e6 : 4e6) && l.values < 9e6 ? kPolicyRows / 2 : kPolicyRows / 4;
    if (requant)
        return l.values < (single ? 3e6 : 4e6) ? kPolicyRows / 4 : l.values < (single ? 6e6 : 14e6) ? kPolicyRows / 2 : kPolicyRows;
    uint32_t tile_rows;
    if (l.half_io)
        tile_rows = l.values < 6.5e6 && rows <= 256 * (int64_t)(kPolicyRows / 4)  ? kPolicyRows / 4
                    : l.values < 25e6 && rows <= 400 * (int64_t)(kPolicyRows / 2) ? kPolicyRows / 2
                    : l.values < 26e6                                             ? kPolicyRows
                                                                                  : kPolicyRowsHalf;
    else if (l.values >= 64e6)
        tile_rows = l.m32 ? kPolicyRows / 4 : fold || l.bits ? kPolicyRows : kPolicyRows / 2;
    else if (single)
        tile_rows = l.values < 3e6 && rows <= 2048 ? kPolicyRows / 4
                    : rows <= 8192 && !(l.bits && l.values >= 6e6) ? kPolicyRows / 2 : kPolicyRows;
    else
        tile_rows = rows <= 256 * (int64_t)(kPolicyRows / 4) && !(l.bits && l.values >= 14e6) ? kPolicyRows / 4
                    : rows <= 400 * (int64_t)(kPolicyRows / 2) ? kPolicyRows / 2 : kPolicyRows;
    const double most = values / kValuesPerRowBlock > 512 ? values / kValuesPerRowBlock : 512;
    while (tile_rows < kPolicyRowsMost && (double)rows > most * tile_rows)
        tile_rows *= 2;
    return tile_rows;
}

// Launches of at most this many values leave the gradient and the second moment's codes in the cache (R1Launch::keep).  The memory-side
// cache holds 256 MB, the gradients of 64M values; the tail of a larger launch still finds its part there.  Steps (us; hint on all loads, then
// without it on these): one to three tensors of 4096 x 4096 65.1 -> 63.0, 122.5 -> 116.8, 174.9 -> 166.4, eight 434.5 -> 427.3;
// 8 bits 78.7 -> 75.7 ... 212.8 -> 199.1; 30 of 512 x 2048 120.9 -> 116.2; GPT-2-XL's set (launches of 210M) 5605 -> 5470; but four
// decoder layers of width 4096 (809M) 2451 -> 2507.  Between the two the line is not sharp: 12 to 32 of 4096 x 4096 (201M to 537M values)
// are the same within 1 % with 4 bits and with an fp32 first moment, and 1 to 2 % faster without the hint at 8 bits.
constexpr double kKeepValues = 256e6;

// The first moment of a record: its codes and scales, or the fp32 moment itself.
static uint8_t *first_moment(const lpmm_nonfused_rank1_tensor &t) { return t.m_codes; }
static float *first_moment_scales(const lpmm_nonfused_rank1_tensor &t) { return t.m_max1; }
static uint8_t *first_moment(const lpmm_rank1_v4bit_tensor &t) { return reinterpret_cast<uint8_t *>(t.m); }
static float *first_moment_scales(const lpmm_rank1_v4bit_tensor &) { return nullptr; }
static uint8_t *first_moment(const lpmm_rank1_mgroup_tensor &t) { return t.m_codes; }
static float *first_moment_scales(const lpmm_rank1_mgroup_tensor &t) { return const_cast<float *>(t.m_max1); }
static float *next_scales(const lpmm_nonfused_rank1_tensor &) { return nullptr; }
static float *next_scales(const lpmm_rank1_v4bit_tensor &) { return nullptr; }
static float *next_scales(const lpmm_rank1_mgroup_tensor &t) { return t.m_max1_next; }

// Tensors that the kernels take as double rows; wraps: as rows of up to 32 too, with any row count (a group then lies in at most two
// tensor rows; the indexes within a row of the matrix have 32 bits).
static bool can_fold_rows(int64_t rows, int64_t cols, bool wraps)
{
    return (cols % kGroup == 64 && rows % 2 == 0) || (wraps && cols % 4 == 0 && (cols >= kGroup || cols == 64) && cols <= (1 << 24));
}

template <int MODE, int FOLD, int N>
static void launch_rank1_passes(const R1LaunchN<N> &l, const float *qmap_m, const float *qmap_v, int passes, hipStream_t stream)
{
    if (passes & 1) {
        const auto update = l.keep ? rank1_update_kernel<MODE, FOLD, true, N> : rank1_update_kernel<MODE, FOLD, false, N>;
        hipLaunchKernelGGL(update, dim3(l.update_tiles), dim3(kThreads), 0, stream, l.update, qmap_m, qmap_v);
    }
    if (passes & 2)
        hipLaunchKernelGGL((rank1_requant_kernel<MODE == kMCodesWide, FOLD, N>), dim3(l.requant_tiles), dim3(kThreads), 0, stream,
                           l.requant, qmap_m, qmap_v);
}

template <int MODE, int N>
static void launch_rank1(const R1LaunchN<N> &l, int folded, const float *qmap_m, const float *qmap_v, int passes, hipStream_t stream)
{
    if constexpr (MODE == kMCodes128)
        if (folded != kNoFold)
            return folded == kDoubles ? launch_rank1_passes<MODE, kDoubles>(l, qmap_m, qmap_v, passes, stream)
                                      : launch_rank1_passes<MODE, kWraps>(l, qmap_m, qmap_v, passes, stream);
    if constexpr (MODE != kMCodes128)
        if (folded != kNoFold)
            return launch_rank1_passes<MODE, kWraps>(l, qmap_m, qmap_v, passes, stream);
    launch_rank1_passes<MODE, kNoFold>(l, qmap_m, qmap_v, passes, stream);
}

// The checks of a call's records.  general: they are for any column count and alignment; can_fold: see rank1_step_multi.
template <int MODE, class Record>
static int check_rank1(const Record *tensors, int64_t count, const float *qmap_m, const float *qmap_v, bool general, bool half_io,
                       bool can_fold, bool wraps = false)
{
    const int64_t real_bytes = general && half_io ? 2 : 4, vec_bytes = general ? real_bytes : 16;
    constexpr bool M32 = MODE == kMFloat;
    LPMM_REQUIRE_PTR(tensors);
    LPMM_REQUIRE_PTR(qmap_m);
    LPMM_REQUIRE_PTR(qmap_v);
    LPMM_REQUIRE_ALIGN(qmap_m, 4);
    LPMM_REQUIRE_ALIGN(qmap_v, 4);
    for (int64_t i = 0; i < count; ++i) {
        const Record &t = tensors[i];
        if (t.rows < 0 || t.cols < 0)
            return LPMM_ERR_SIZE;
        if (!general && t.cols % (MODE == kMCodesWide && !can_fold ? 8 : kGroup) != 0 && !(can_fold && can_fold_rows(t.rows, t.cols, wraps)))
            return LPMM_ERR_SIZE;
        if (t.rows == 0 || t.cols == 0)
            continue;
        const int64_t col_blocks = (t.cols + kGroup - 1) / kGroup;
        // an upper bound: tiles hold at least 16 rows, the last group adds fewer than `resident` blocks
        const int64_t row_blocks = (t.rows + kDppRows - 1) / kDppRows + kPolicyResident;
        if (col_blocks > 0x7fffffffLL / 2 || row_blocks > 0x7fffffffLL / col_blocks ||
            t.rows > INT64_MAX / t.cols)
            return LPMM_ERR_SIZE;
        LPMM_REQUIRE_PTR(t.p);
        LPMM_REQUIRE_PTR(t.g);
        LPMM_REQUIRE_PTR(first_moment(t));
        if (!M32)
            LPMM_REQUIRE_PTR(first_moment_scales(t));
        LPMM_REQUIRE_PTR(t.v_codes);
        LPMM_REQUIRE_PTR(t.v_rowmax);
        LPMM_REQUIRE_PTR(t.v_colmax);
        LPMM_REQUIRE_PTR(t.v_rowmax_next);
        LPMM_REQUIRE_PTR(t.v_colmax_next);
        LPMM_REQUIRE_ALIGN(t.p, vec_bytes);
        LPMM_REQUIRE_ALIGN(t.g, vec_bytes);
        LPMM_REQUIRE_ALIGN(first_moment(t), M32 && !general ? 16 : 4);
        LPMM_REQUIRE_ALIGN(t.v_codes, 4);
        LPMM_REQUIRE_ALIGN(first_moment_scales(t), real_bytes);
        if (MODE == kMCodesWide) {
            LPMM_REQUIRE_PTR(next_scales(t));
            LPMM_REQUIRE_ALIGN(next_scales(t), 4);
            if (next_scales(t) == first_moment_scales(t))
                return LPMM_ERR_ARG;
        }
        LPMM_REQUIRE_ALIGN(t.v_rowmax, real_bytes);
        LPMM_REQUIRE_ALIGN(t.v_colmax, vec_bytes);
        LPMM_REQUIRE_ALIGN(t.v_rowmax_next, 4);
        LPMM_REQUIRE_ALIGN(t.v_colmax_next, general ? 4 : 16);
        if (t.v_rowmax == t.v_rowmax_next || t.v_colmax == t.v_colmax_next)
            return LPMM_ERR_ARG;
    }
    return LPMM_OK;
}

// Where the launch that begins with tensors[i] ends: after `most` tensors that are not empty, or, from 48M values on, where the first of
// the tensors that wrap meets others or the other way round, double rows among the others.  4-bit first moments in groups of 128: the kernel
// for both takes 1 to 3 % longer than the others' own, so that a large launch holds one kind (GPT-2-XL's
// 50257 x 1600 embedding with 31 of its matrices, and too large a launch for the cache: 5255 -> 5207 us a step).  A launch
// of its own for a few small ones would cost more.  The other first moments have no kernel of their own for double rows, and there the line is no
// better and no worse than one between kernels (double rows among those that wrap).  Steps with this one -> that one, fp32 / 8 bits / groups of 256: eight of
// 4096 x 4096, then eight of 4096 x 4160 1163 / 995 / 961 -> 1120 / 975 / 921, but four, then two 424 / 367 / 355 -> 426 / 381 / 349; four of 4096 x
// 4160, then two of 4096 x 4100 443 / 387 / 384 -> 431 / 378 / 371, but eight of each (beyond the cache) 1140 / 996 / 973 -> 1166 / 1009 / 1003.
template <class Record>
static int64_t launch_end(const Record *tensors, int64_t i, int64_t count, int most, bool can_fold)
{
    const auto wraps = [&](const Record &t) { return can_fold && t.cols % kGroup != 0 && !can_fold_rows(t.rows, t.cols, false); };
    double values = 0;
    int k = 0;
    bool any_wraps = false, any_other = false;
    for (; i < count && k < most; ++i) {
        const Record &t = tensors[i];
        if (t.rows == 0 || t.cols == 0)
            continue;
        const bool w = wraps(t);
        if (values >= 48e6 && (w ? !any_wraps : !any_other))
            break;
        any_wraps = any_wraps || w;
        any_other = any_other || !w;
        values += (double)t.rows * (double)t.cols;
        ++k;
    }
    return i;
}

// Validation, batching into launches of at most kR1Max tensors (4-bit codes of both moments: kR1Many small ones), and the launches.
// m_lg: the first moment's group holds 128 << m_lg values (MODE kMCodesWide only).
// folds: a record per tensor, of ndim 0 where the tensor is a matrix (lpmm_nonfused_adamw4bit_rank1_nd_step_multi).
// plain: tensors with fp32 states that go with the clearing, as many as its launches take.  wraps: see can_fold_rows.
template <int MODE, class Record>
static int rank1_step_multi(const Record *tensors, int64_t count, const float *qmap_m, const float *qmap_v,
                            uint32_t m_lg, double beta1, double beta2, double lr, double weight_decay, double eps,
                            void *stream, int bits_m = 4, int bits_v = 4, const void *table_m = nullptr,
                            const void *table_v = nullptr, int passes = 3, bool half_io = false, const NewCodes *out = nullptr,
                            const lpmm_rank1_small_vector *folds = nullptr, PlainSet *plain = nullptr, bool wraps = false)
{
    // passes: 1 = the first pass alone (with the clearing of the next statistics), 2 = the second alone,
    // 3 = both; one at a time only where the launches below are this file's own, or general ones: any column count,
    // any alignment (nonfused_rank1_any.hip; wide-group and fp32 records, at most one launch's worth, none empty, checked by the caller).
    const bool general = out != nullptr;
    if (passes < 1 || passes > 3 || (passes != 3 && !general && (MODE != kMCodes128 || bits_m != 4 || half_io)))
        return LPMM_ERR_ARG;
    constexpr bool M32 = MODE == kMFloat;
    // 4-bit codes in 128-value groups: a column count of 64 modulo 128 with an even row count is
    // served as double rows (rank1_tiles.hpp)
    // (byte codes, fp32 first moments and wide groups: as rows of any number, where the caller may)
    const bool can_fold = !half_io && !general && (wraps || (MODE == kMCodes128 && bits_m == 4));
    if (count < 0)
        return LPMM_ERR_SIZE;
    if (count == 0)
        return LPMM_OK;
    if (!general) {
        const int bad = check_rank1<MODE>(tensors, count, qmap_m, qmap_v, false, half_io, can_fold, wraps);
        if (bad != LPMM_OK)
            return bad;
    }
    // column counts that are no multiple of 128 (wide-group records only) and do not fold: every tensor of the call
    // then takes the kernels for ragged rows
    bool ragged = false;
    for (int64_t i = 0; i < count; ++i)
        ragged = ragged || (MODE == kMCodesWide && tensors[i].cols % kGroup != 0 && !can_fold);

    hipStream_t s = (hipStream_t)stream;
    if (passes & 1) {
        ClearRanges<kClearMax> ranges;
        int n = 0;
        int64_t longest = 0;
        const auto launch_clear = [&] {
            const int64_t blocks = (longest + kThreads - 1) / kThreads;
            const dim3 grid((uint32_t)(blocks > 64 ? 64 : blocks), (uint32_t)n);
            if (n != 0 && plain != nullptr && plain->next < plain->count)
                launch_clear_plain(ranges, n, grid.x, *plain, beta1, beta2, lr, weight_decay, eps, s);
            else if (n > kClearFew)
                hipLaunchKernelGGL(rank1_clear_kernel<kClearMax>, grid, dim3(kThreads), 0, s, ranges);
            else if (n != 0)
                hipLaunchKernelGGL(rank1_clear_kernel<kClearFew>, grid, dim3(kThreads), 0, s, ranges_from<kClearFew>(ranges));
            n = 0;
            longest = 0;
        };
        const int most = plain != nullptr && plain->next < plain->count ? kClearJoined : kClearMax;
        const auto clear = [&](float *at, int64_t count_of) {
            if (n != 0 && ranges.at[n - 1] + ranges.n[n - 1] == at) {
                ranges.n[n - 1] += count_of;
            } else {
                if (n == most)
                    launch_clear();
                ranges.at[n] = at;
                ranges.n[n++] = count_of;
            }
            longest = ranges.n[n - 1] > longest ? ranges.n[n - 1] : longest;
        };
        const int64_t group = (int64_t)kGroup << m_lg;
        for (int64_t i = 0; i < count; ++i) {
            const Record &t = tensors[i];
            if (t.rows == 0 || t.cols == 0)
                continue;
            clear(t.v_rowmax_next, t.rows);
            clear(t.v_colmax_next, t.cols);
            if (next_scales(t) != nullptr)
                clear(next_scales(t), (t.rows * t.cols + group - 1) / group);
        }
        launch_clear();
        const int st = launch_status();
        if (st != LPMM_OK)
            return st;
    }

    const NfHyper c = make_nf_hyper(beta1, beta2, lr, weight_decay, eps, 1.0);
    NfHypers hypers(beta1, beta2, lr, weight_decay, eps);
    int64_t i = 0;
    // one launch's worth of tensors from i on
    const auto launch = [&](auto &l) -> int {
        constexpr int kMost = std::decay_t<decltype(l)>::kMax;
        auto &args = l.update;
        args.decay = c.decay;
        args.w1 = c.w1;
        args.b2 = c.b2;
        args.w2 = c.w2;
        args.eps = c.eps;
        int k = 0;
        const int64_t end = launch_end(tensors, i, count, kMost, can_fold);
        // what this launch will hold decides its tiles' rows
        LaunchKind kind = {half_io, M32, bits_m != 4, 0, {false, false}};
        const auto each = [&](auto &&f) {
            for (int64_t j = i; j < end; ++j)
                if (tensors[j].rows != 0 && tensors[j].cols != 0)
                    f(tensors[j]);
        };
        int held = 0;
        each([&](const Record &t) {
            kind.values += (double)t.rows * (double)t.cols;
            ++held;
        });
        if (general || half_io || held == 1) {
            uint64_t blocks[2] = {0, 0};
            each([&](const Record &t) {
                const Matrix m = matrix_of(t.rows, t.cols, can_fold);
                for (int pass = 0; pass < 2; ++pass) {
                    const Blocks b = blocks_of(m.rows, m.col_blocks, pass_rows_policy(kind, pass == 1, m, t.cols & 1));
                    blocks[pass] += b.rows * b.col_tiles;
                }
            });
            kind.spread[0] = blocks[0] < kSpreadBelow;
            kind.spread[1] = blocks[1] < kSpreadBelow;
        }
        uint64_t tiles = 0, tiles2 = 0;
        uint32_t start2[kMost + 1] = {0};
        TileShape shape2[kMost];
        float *scale2[kMost];  // the column statistics of the second pass
        const lpmm_rank1_small_vector *between[kMost];
        int betweens = 0;
        int folded = kNoFold;  // what the launch's tensors need
        args.tile_start[0] = 0;
        while (i < end) {
            const Record &t = tensors[i];
            if (t.rows == 0 || t.cols == 0) {
                ++i;
                continue;
            }
            const uint32_t col_blocks = (uint32_t)((t.cols + kGroup - 1) / kGroup);
            TensorR1 &d = args.t[k];
            const Matrix m = matrix_of(t.rows, t.cols, can_fold);
            const bool odd = t.cols & 1;
            const uint64_t nt = shape_tiles(m.rows, m.col_blocks, d.tile, pass_rows_policy(kind, false, m, odd),
                                            kind.spread[0]);
            const uint64_t nt2 = shape_tiles(m.rows, m.col_blocks, shape2[k], pass_rows_policy(kind, true, m, odd),
                                             kind.spread[1]);
            if (tiles + nt > 0x7fffffffULL || tiles2 + nt2 > 0x7fffffffULL)
                break;
            d.p = t.p;
            d.g = t.g;
            d.mc = first_moment(t);
            d.ms = first_moment_scales(t);
            d.ms_new = next_scales(t);
            d.m_lg = m_lg;
            d.vc = t.v_codes;
            d.row_old = t.v_rowmax;
            d.col_old = t.v_colmax;
            d.row_new = t.v_rowmax_next;
            d.col_new = t.v_colmax_next;
            d.rows = t.rows;
            d.col_blocks = col_blocks;
            d.col_tail = (uint32_t)(t.cols - (int64_t)(col_blocks - 1) * kGroup);
            // what the kernels for any column count took before
            d.tile.drop_nan = shape2[k].drop_nan =
                m.lg != 0 && (M32 || bits_m != 4 || (!can_fold_rows(t.rows, t.cols, false) && (t.cols % 8 != 0 || (folds != nullptr && folds[i].ndim != 0))));
            const NfHyper &h = hypers.at(t.step);
            d.neg_step_size = h.neg_step_size;
            d.bc2_sqrt = h.bc2_sqrt;
            d.rbc2_sqrt = h.rbc2_sqrt;
            tiles += nt;
            tiles2 += nt2;
            if (m.lg != 0)
                folded = std::max(folded, (int)(can_fold_rows(t.rows, t.cols, false) ? kDoubles : kWraps));
            scale2[k] = d.col_new;
            if (folds != nullptr && folds[i].ndim != 0) {
                scale2[k] = folds[i].scale;
                between[betweens++] = folds + i;
            }
            args.tile_start[++k] = (uint32_t)tiles;
            start2[k] = (uint32_t)tiles2;
            ++i;
        }
        if (k == 0) {
            if (i < end)
                return LPMM_ERR_SIZE;  // a single tensor with more tiles than a grid holds
            return LPMM_OK;
        }
        args.count = k;
        for (int j = k + 1; j <= kMost; ++j) {
            args.tile_start[j] = (uint32_t)tiles;
            start2[j] = (uint32_t)tiles2;
        }
        l.requant = args;
        for (int j = 0; j < k; ++j) {
            l.requant.t[j].tile = shape2[j];
            l.requant.t[j].col_new = scale2[j];
        }
        memcpy(l.requant.tile_start, start2, sizeof start2);
        l.update_tiles = (uint32_t)tiles;
        l.requant_tiles = (uint32_t)tiles2;
        l.keep = kind.values <= kKeepValues;
        if constexpr (kMost == kR1Max) {
            if (general) {
                const AnyKind any = half_io ? kAnyHalf : M32 ? kAnyFloatM : bits_m != 4 ? kAnyBits : kAnyCodes4;
                launch_rank1_any(l, *out, qmap_m, qmap_v, any, bits_m, bits_v, static_cast<const uint32_t *>(table_m),
                                 static_cast<const uint32_t *>(table_v), passes, s);
                return launch_status();
            }
            if (half_io) {
                launch_rank1_half(l, qmap_m, qmap_v, s);
                return launch_status();
            }
            if (ragged || (MODE == kMCodesWide && m_lg == 0 && folded == kNoFold)) {
                launch_rank1_ragged(l, qmap_m, qmap_v, s);
                return launch_status();
            }
            if (bits_m != 4) {
                launch_rank1_bits(l, folded != kNoFold, qmap_m, qmap_v, bits_m, bits_v, static_cast<const uint32_t *>(table_m),
                                  static_cast<const uint32_t *>(table_v), s);
                return launch_status();
            }
        }
        if (betweens != 0) {
            launch_rank1<MODE>(l, folded, qmap_m, qmap_v, 1, s);
            const int st = launch_small_vectors(between, betweens, s);
            if (st != LPMM_OK)
                return st;
            launch_rank1<MODE>(l, folded, qmap_m, qmap_v, 2, s);
        } else {
            launch_rank1<MODE>(l, folded, qmap_m, qmap_v, passes, s);
        }
        return launch_status();
    };
    // More tensors a launch where they are small: a launch's start and end, 8 to 10 us of both passes, are then a good part of it.
    // Steps with 32 -> 64 a launch: 64 of 512 x 512 71.5 -> 67, of 800 x 1024 (52M values) 187 -> 174, of 1024 x 1024 229.5 -> 221, of 1024 x
    // 2048 426 -> 422; 128 of 448 x 448 132 -> 120, of 192 x 128 x 3 x 3 156 -> 140; from 200M values on nothing, from 270M on 1 to 2 %
    // slower: the second pass finds less of what the first has read.
    constexpr double kManyValues = 80e6;
    const bool own_kernels = MODE == kMCodes128 && !general && !half_io && bits_m == 4;
    R1Launch l;
    R1LaunchN<kR1Many> many;
    while (i < count) {
        double values = 0;
        int held = 0;
        for (int64_t j = i; own_kernels && j < count && held < kR1Many; ++j)
            if (tensors[j].rows != 0 && tensors[j].cols != 0) {
                values += (double)tensors[j].rows * (double)tensors[j].cols;
                ++held;
            }
        int st;
        if constexpr (MODE == kMCodes128)
            st = held > kR1Max && values <= kManyValues ? launch(many) : launch(l);
        else
            st = launch(l);
        if (st != LPMM_OK)
            return st;
    }
    return LPMM_OK;
}

extern "C" int lpmm_nonfused_adamw4bit_rank1_step_multi(const lpmm_nonfused_rank1_tensor *tensors, int64_t count,
                                                        const float *qmap_m, const float *qmap_v, double beta1,
                                                        double beta2, double lr, double weight_decay,
                                                        double eps, void *stream)
{
    return rank1_step_multi<kMCodes128>(tensors, count, qmap_m, qmap_v, 0, beta1, beta2, lr, weight_decay, eps, stream);
}

int lpmm::rank1_step_multi_half(const lpmm_nonfused_rank1_tensor *tensors, int64_t count, const float *qmap_m,
                                const float *qmap_v, double beta1, double beta2, double lr, double weight_decay,
                                double eps, void *stream)
{
    return rank1_step_multi<kMCodes128>(tensors, count, qmap_m, qmap_v, 0, beta1, beta2, lr, weight_decay, eps, stream,
                                        4, 4, nullptr, nullptr, 3, true);
}

extern "C" int lpmm_nonfused_adamw4bit_rank1_pass_multi(const lpmm_nonfused_rank1_tensor *tensors, int64_t count,
                                                        const float *qmap_m, const float *qmap_v, double beta1,
                                                        double beta2, double lr, double weight_decay,
                                                        double eps, int pass, void *stream)
{
    if (pass != 1 && pass != 2)
        return LPMM_ERR_ARG;
    return rank1_step_multi<kMCodes128>(tensors, count, qmap_m, qmap_v, 0, beta1, beta2, lr, weight_decay, eps, stream,
                                        4, 4, nullptr, nullptr, pass);
}

static int nd_step_multi(const lpmm_nonfused_rank1_tensor *tensors, const lpmm_rank1_small_vector *folds, int64_t count,
                         const float *qmap_m, const float *qmap_v, double beta1, double beta2, double lr, double weight_decay, double eps,
                         void *stream, PlainSet *plain)
{
    if (count < 0)
        return LPMM_ERR_SIZE;
    if (count == 0)
        return LPMM_OK;
    LPMM_REQUIRE_PTR(tensors);
    LPMM_REQUIRE_PTR(folds);
    for (int64_t i = 0; i < count; ++i) {
        const lpmm_rank1_small_vector &v = folds[i];
        if (v.ndim == 0 || tensors[i].rows == 0 || tensors[i].cols == 0)
            continue;
        const int bad = check_small_vectors(&v, 1);
        if (bad != LPMM_OK)
            return bad;
        int64_t n = 1;
        for (int k = 0; k < v.ndim; ++k)
            n *= v.shape[k];
        if (n != tensors[i].cols)
            return LPMM_ERR_SIZE;
        if (v.x != tensors[i].v_colmax_next || v.scale == v.x || v.scale == tensors[i].v_colmax)
            return LPMM_ERR_ARG;
        LPMM_REQUIRE_ALIGN(v.scale, 16);
    }
    return rank1_step_multi<kMCodes128>(tensors, count, qmap_m, qmap_v, 0, beta1, beta2, lr, weight_decay, eps, stream, 4, 4, nullptr,
                                        nullptr, 3, false, nullptr, folds, plain, true);
}

extern "C" int lpmm_nonfused_adamw4bit_rank1_nd_step_multi(const lpmm_nonfused_rank1_tensor *tensors,
                                                           const lpmm_rank1_small_vector *folds, int64_t count, const float *qmap_m,
                                                           const float *qmap_v, double beta1, double beta2, double lr,
                                                           double weight_decay, double eps, void *stream)
{
    return nd_step_multi(tensors, folds, count, qmap_m, qmap_v, beta1, beta2, lr, weight_decay, eps, stream, nullptr);
}

extern "C" int lpmm_nonfused_adamw_v4bit_rank1_step_multi(const lpmm_rank1_v4bit_tensor *tensors, int64_t count,
                                                          const float *qmap_v, double beta1, double beta2,
                                                          double lr, double weight_decay, double eps,
                                                          void *stream)
{
    // the update kernel keeps the second moment's map in both map slots; only the second is read
    return rank1_step_multi<kMFloat>(tensors, count, qmap_v, qmap_v, 0, beta1, beta2, lr, weight_decay, eps, stream);
}

extern "C" int lpmm_nonfused_adamw4bit_rank1_mgroup_step_multi(const lpmm_rank1_mgroup_tensor *tensors, int64_t count,
                                                               const float *qmap_m, const float *qmap_v,
                                                               int64_t m_group_size, double beta1, double beta2,
                                                               double lr, double weight_decay, double eps,
                                                               void *stream)
{
    uint32_t m_lg = 0;
    while (m_lg < 5 && ((int64_t)kGroup << m_lg) < m_group_size)
        ++m_lg;
    if (((int64_t)kGroup << m_lg) != m_group_size)
        return LPMM_ERR_SIZE;  // 128, 256, 512, 1024, 2048 or 4096
    return rank1_step_multi<kMCodesWide>(tensors, count, qmap_m, qmap_v, m_lg, beta1, beta2, lr, weight_decay, eps,
                                         stream);
}

extern "C" int lpmm_nonfused_adamw_bits_rank1_step_multi(const lpmm_nonfused_rank1_tensor *tensors, int64_t count,
                                                         const float *qmap_m, int bits_m, const float *qmap_v,
                                                         int bits_v, double beta1, double beta2, double lr,
                                                         double weight_decay, double eps, void *stream)
{
    return lpmm_nonfused_adamw_bits_rank1_step_multi_table(tensors, count, qmap_m, bits_m, nullptr, qmap_v, bits_v,
                                                           nullptr, beta1, beta2, lr, weight_decay, eps, stream);
}

extern "C" int lpmm_nonfused_adamw_bits_rank1_step_multi_table(const lpmm_nonfused_rank1_tensor *tensors, int64_t count,
                                                               const float *qmap_m, int bits_m, const void *table_m,
                                                               const float *qmap_v, int bits_v, const void *table_v,
                                                               double beta1, double beta2, double lr,
                                                               double weight_decay, double eps, void *stream)
{
    if (bits_m < 5 || bits_m > 8 || bits_v < 5 || bits_v > 8)
        return LPMM_ERR_ARG;  // the widths that store one code per byte
    if (table_m != nullptr)
        LPMM_REQUIRE_ALIGN(table_m, 16);
    if (table_v != nullptr)
        LPMM_REQUIRE_ALIGN(table_v, 16);
    return rank1_step_multi<kMCodes128>(tensors, count, qmap_m, qmap_v, 0, beta1, beta2, lr, weight_decay, eps, stream,
                                        bits_m, bits_v, table_m, table_v);
}

// A launch's worth of records for any column count in the two forms that rank1_step_multi takes.
struct AnyRecords {
    lpmm_rank1_mgroup_tensor wide[kR1Max];
    lpmm_rank1_v4bit_tensor plain[kR1Max];  // fp32 first moment

    void set(int k, const lpmm_rank1_any_tensor &t)
    {
        lpmm_rank1_mgroup_tensor &w = wide[k];
        lpmm_rank1_v4bit_tensor &f = plain[k];
        f.p = w.p = static_cast<float *>(t.p);
        f.g = w.g = static_cast<const float *>(t.g);
        f.m = static_cast<float *>(t.m);
        w.m_codes = static_cast<uint8_t *>(t.m);
        w.m_max1 = static_cast<const float *>(t.m_max1);
        w.m_max1_next = static_cast<float *>(t.m_max1_next);
        f.v_codes = w.v_codes = const_cast<uint8_t *>(t.v_codes);
        f.v_rowmax = w.v_rowmax = static_cast<const float *>(t.v_rowmax);
        f.v_colmax = w.v_colmax = static_cast<const float *>(t.v_colmax);
        f.v_rowmax_next = w.v_rowmax_next = static_cast<float *>(t.v_rowmax_next);
        f.v_colmax_next = w.v_colmax_next = static_cast<float *>(t.v_colmax_next);
        f.rows = w.rows = t.rows;
        f.cols = w.cols = t.cols;
        f.step = w.step = t.step;
        f.reserved = w.reserved = 0.0f;
    }
};

// All records of a call, before the first launch: a call with an invalid one changes nothing.
static int check_any(const lpmm_rank1_any_tensor *tensors, int64_t count, AnyKind kind, const float *qmap_m, const float *qmap_v)
{
    for (int64_t i = 0; i < count; ++i) {
        const lpmm_rank1_any_tensor &t = tensors[i];
        if (t.rows == 0 || t.cols == 0)
            continue;
        LPMM_REQUIRE_PTR(t.v_codes_next);
        LPMM_REQUIRE_ALIGN(t.v_codes_next, 4);
        if (t.v_codes_next == t.v_codes)
            return LPMM_ERR_ARG;
        if (kind != kAnyFloatM) {
            LPMM_REQUIRE_PTR(t.m_codes_next);
            LPMM_REQUIRE_ALIGN(t.m_codes_next, 4);
            if (t.m_codes_next == t.m)
                return LPMM_ERR_ARG;
        }
    }
    AnyRecords one;
    for (int64_t i = 0; i < count; ++i) {
        if (tensors[i].rows == 0 || tensors[i].cols == 0)
            continue;
        one.set(0, tensors[i]);
        const int bad = kind == kAnyFloatM
                            ? check_rank1<kMFloat>(one.plain, 1, qmap_v, qmap_v, true, false, false)
                            : check_rank1<kMCodesWide>(one.wide, 1, qmap_m, qmap_v, true, kind == kAnyHalf, false);
        if (bad != LPMM_OK)
            return bad;
    }
    return LPMM_OK;
}

int lpmm::rank1_any_step_multi(const lpmm_rank1_any_tensor *tensors, int64_t count, AnyKind kind, uint32_t m_lg,
                               const float *qmap_m, int bits_m, const void *table_m, const float *qmap_v, int bits_v,
                               const void *table_v, double beta1, double beta2, double lr, double weight_decay, double eps,
                               int passes, void *stream, PlainSet *plain)
{
    const int bad = check_any(tensors, count, kind, qmap_m, qmap_v);
    if (bad != LPMM_OK)
        return bad;
    AnyRecords rec;
    NewCodes out;
    // First the tensors that go in runs of four values, then the others: a launch holds one kind.  Where a call has both, the second
    // set of launches (about 30 us: three layers of width 64 and 218 in float16 90 -> 124 us a step) has to be worth it: runs save about
    // 1.5 us per million values.
    double run_values = 0;
    bool mixed = false;
    for (int64_t i = 0; i < count; ++i) {
        if (rank1_any_runs(tensors[i], kind))
            run_values += (double)tensors[i].rows * (double)tensors[i].cols;
        else
            mixed = mixed || (tensors[i].rows != 0 && tensors[i].cols != 0);
    }
    const bool use_runs = !mixed || run_values >= 24e6;
    for (int side = 0; side < 2; ++side) {
        for (int64_t i = 0; i < count;) {
            int k = 0;
            out.runs = side == 0;
            for (; i < count && k < kR1Max; ++i) {
                const lpmm_rank1_any_tensor &t = tensors[i];
                if (t.rows == 0 || t.cols == 0 || (use_runs && rank1_any_runs(t, kind)) != out.runs)
                    continue;
                rec.set(k, t);
                out.v[k] = t.v_codes_next;
                out.m[k++] = t.m_codes_next;
            }
            const int st = kind == kAnyFloatM
                               ? rank1_step_multi<kMFloat>(rec.plain, k, qmap_v, qmap_v, 0, beta1, beta2, lr, weight_decay, eps, stream, 4,
                                                           4, nullptr, nullptr, passes, false, &out, nullptr, plain)
                               : rank1_step_multi<kMCodesWide>(rec.wide, k, qmap_m, qmap_v, m_lg, beta1, beta2, lr, weight_decay, eps,
                                                               stream, bits_m, bits_v, table_m, table_v, passes, kind == kAnyHalf, &out,
                                                               nullptr, plain);
            if (st != LPMM_OK)
                return st;
        }
    }
    return LPMM_OK;
}

extern "C" int lpmm_nonfused_adamw_rank1_any_step_multi(const lpmm_rank1_any_tensor *tensors, int64_t count, int kind,
                                                        int64_t m_group_size, const float *qmap_m, int bits_m,
                                                        const void *table_m, const float *qmap_v, int bits_v,
                                                        const void *table_v, double beta1, double beta2, double lr,
                                                        double weight_decay, double eps, int passes, void *stream)
{
    if (count < 0)
        return LPMM_ERR_SIZE;
    if (count == 0)
        return LPMM_OK;
    LPMM_REQUIRE_PTR(tensors);
    if (kind < LPMM_RANK1_CODES4 || kind > LPMM_RANK1_HALF || passes < 1 || passes > 3)
        return LPMM_ERR_ARG;
    const bool bytes = kind == LPMM_RANK1_CODES8;
    if (bytes ? bits_m < 5 || bits_m > 8 || bits_v < 5 || bits_v > 8 : bits_m != 4 || bits_v != 4)
        return LPMM_ERR_ARG;
    if (table_m != nullptr)
        LPMM_REQUIRE_ALIGN(table_m, 16);
    if (table_v != nullptr)
        LPMM_REQUIRE_ALIGN(table_v, 16);
    uint32_t m_lg = 0;
    while (m_lg < 5 && ((int64_t)kGroup << m_lg) < m_group_size)
        ++m_lg;
    if (((int64_t)kGroup << m_lg) != m_group_size || (m_lg != 0 && kind != LPMM_RANK1_CODES4))
        return LPMM_ERR_SIZE;  // 128; 4-bit codes also 256, 512, 1024, 2048, 4096
    if (kind == LPMM_RANK1_HALF)
        return passes == 3 ? rank1_any_half(tensors, count, qmap_m, qmap_v, beta1, beta2, lr, weight_decay, eps, stream)
                           : LPMM_ERR_ARG;
    return rank1_any_step_multi(tensors, count, (AnyKind)kind, m_lg, qmap_m, bits_m, table_m, qmap_v, bits_v, table_v, beta1,
                                beta2, lr, weight_decay, eps, passes, stream);
}

// 128 << lg, or -1
static int lg_of_group(int64_t m_group_size)
{
    for (int lg = 0; lg <= 5; ++lg)
        if (((int64_t)kGroup << lg) == m_group_size)
            return lg;
    return -1;
}

extern "C" int lpmm_nonfused_rank1_fp32_step_multi(int kind, const void *tensors, const lpmm_rank1_small_vector *folds, int64_t count,
                                                   const lpmm_adamw_fp32_tensor *plain, int64_t plain_count, int64_t m_group_size,
                                                   const float *qmap_m, int bits_m, const void *table_m, const float *qmap_v, int bits_v,
                                                   const void *table_v, double beta1, double beta2, double lr, double weight_decay,
                                                   double eps, void *stream)
{
    if (count < 0 || plain_count < 0)
        return LPMM_ERR_SIZE;
    if (plain_count != 0) {
        const int bad = check_fp32(plain, plain_count, 4);
        if (bad != LPMM_OK)
            return bad;
    }
    const bool bytes = kind == LPMM_STEP_BITS || kind == LPMM_STEP_ANY + LPMM_RANK1_CODES8;
    if (bytes ? bits_m < 5 || bits_m > 8 || bits_v < 5 || bits_v > 8 : bits_m != 4 || bits_v != 4)
        return LPMM_ERR_ARG;
    if (table_m != nullptr)
        LPMM_REQUIRE_ALIGN(table_m, 16);
    if (table_v != nullptr)
        LPMM_REQUIRE_ALIGN(table_v, 16);
    const int m_lg = lg_of_group(m_group_size);
    if (m_lg < 0 || (m_lg != 0 && kind != LPMM_STEP_GROUPS && kind != LPMM_STEP_GROUPS_WRAP && kind != LPMM_STEP_ANY + LPMM_RANK1_CODES4))
        return LPMM_ERR_SIZE;
    PlainSet set = {plain, plain_count, 0};
    const auto matrices = static_cast<const lpmm_nonfused_rank1_tensor *>(tensors);
    int st = LPMM_OK;
    if (count != 0) {
        LPMM_REQUIRE_PTR(tensors);
        switch (kind) {
        case LPMM_STEP_MATRIX:
        case LPMM_STEP_BITS:
            st = rank1_step_multi<kMCodes128>(matrices, count, qmap_m, qmap_v, 0, beta1, beta2, lr, weight_decay, eps, stream, bits_m,
                                              bits_v, table_m, table_v, 3, false, nullptr, nullptr, &set, true);
            break;
        case LPMM_STEP_ND:
            st = nd_step_multi(matrices, folds, count, qmap_m, qmap_v, beta1, beta2, lr, weight_decay, eps, stream, &set);
            break;
        case LPMM_STEP_FLOAT_M:
            st = rank1_step_multi<kMFloat>(static_cast<const lpmm_rank1_v4bit_tensor *>(tensors), count, qmap_v, qmap_v, 0, beta1, beta2,
                                           lr, weight_decay, eps, stream, 4, 4, nullptr, nullptr, 3, false, nullptr, nullptr, &set, true);
            break;
        case LPMM_STEP_GROUPS:
        case LPMM_STEP_GROUPS_WRAP:
            st = rank1_step_multi<kMCodesWide>(static_cast<const lpmm_rank1_mgroup_tensor *>(tensors), count, qmap_m, qmap_v,
                                               (uint32_t)m_lg, beta1, beta2, lr, weight_decay, eps, stream, 4, 4, nullptr, nullptr, 3,
                                               false, nullptr, nullptr, &set, kind == LPMM_STEP_GROUPS_WRAP);
            break;
        case LPMM_STEP_ANY + LPMM_RANK1_CODES4:
        case LPMM_STEP_ANY + LPMM_RANK1_FLOAT_M:
        case LPMM_STEP_ANY + LPMM_RANK1_CODES8:
            st = rank1_any_step_multi(static_cast<const lpmm_rank1_any_tensor *>(tensors), count, (AnyKind)(kind - LPMM_STEP_ANY),
                                      (uint32_t)m_lg, qmap_m, bits_m, table_m, qmap_v, bits_v, table_v, beta1, beta2, lr, weight_decay,
                                      eps, 3, stream, &set);
            break;
        default:
            return LPMM_ERR_ARG;
        }
    }
    return st != LPMM_OK ? st
                         : lpmm_nonfused_update_multi(plain + set.next, plain_count - set.next, beta1, beta2, lr, weight_decay, eps, stream);
}
