// AdamW steps on float16 parameters with 4-bit states: the non-fused step as one pass (block-wise second
// moment) and as two passes (rank-1 second moment), and the fused operator's half instantiation (the
// one-pass kernel with that operator's arithmetic and layout, adamw4bit_half_kernel<true>).
//
// With fused=False the reference runs its chain of PyTorch ops in the parameters' type
// (lpmm/optim/adamw.py:367-369, :394-434): every op converts its half operands to float, computes as
// the float kernel does and rounds the result to half once; Python scalars enter as floats.  States,
// scales and statistics are half tensors (lpmm/functional.py:184-203); the normalised values are
// rounded to half by the division and widened to float again by the pack kernel before the search
// (lpmm/cpp_extension/quantization_kernel.cu:450); the unpacked map value (float) times the half scale
// is a float product that takes the state's type last (lpmm/functional.py:97-118, :150).  The kernels
// below do that arithmetic in registers, with a rounding to half wherever an op of the chain ends,
// and move 8.06 bytes per parameter (block-wise second moment: p 2 + 2, g 2, codes 1 + 1, scales
// 4 * 2 / 128) or 7.52 + 3 bytes (rank-1 second moment) instead of the chain's 50.
//
// Layouts, tiles and statistics are those of the float kernels (nonfused_m32.hip, nonfused_rank1_bits.hip).
// The maxima of the new second moment over rows and columns are taken with integer atomics on the
// float images of the half values in a float work array (a maximum of half values is a half value);
// a last small kernel writes them out as halfs.
//
// Arithmetic bounds the one pass and the update (eleven roundings per element), so what counts is
// instructions per element.  Halfs stay in pairs, roundings are packed, products read halfs directly (lpmm_half.hpp), two codes
// are decoded by one read and the normalised halfs encoded as halfs, maxima over a lane's columns stay in registers through its
// passes instead of going to LDS one by one, and addresses advance by one addition each.  Kernels of the usual constants (USUAL)
// have no branch in the chain.  VALU instructions an element, before and after the decoding, encoding and roots of halfs: update 48 -> 37,
// second pass 19 -> 14.  Four decoder layers of width 4096 (8.1e8 values), a step: 1737 -> 1570 us (the memory system's: 1360);
// the one pass on a LLaMA-7B-shaped set (6.7e9 values) 13.4 -> 11.3 ms a step.  Six waves per SIMD for the update: within 1 % of four,
// five and seven.
#include "lpmm_half.hpp"

namespace lpmm {

// ---------------------------------------------------------------------------------------
// One pass: both moments block-wise over 128 values.
// ---------------------------------------------------------------------------------------
constexpr int kHTile = kThreads * kEltsPerLane;  // 2048 = one pack group
constexpr int kHMax = 48;                        // tensors per launch
static_assert(kHTile == LPMM_PACK_GROUP, "a tile is a pack group of the non-fused layout");

struct TensorH {
    h16 *p;
    const h16 *g;
    uint8_t *mc, *vc;
    h16 *ms, *vs;
    int64_t n;
    float neg_step_size, bc2_sqrt, rbc2_sqrt;
    uint32_t vec;  // p and g allow 8-byte accesses
};

struct MultiH {
    TensorH t[kHMax];
    uint32_t tile_start[kHMax + 1];
    float decay, w1, b2, w2, eps;
};
static_assert(sizeof(MultiH) + sizeof(Hyper) + 2 * sizeof(void *) <= 4096, "kernel arguments exceed 4 KB");
static_assert(kHMax <= kWave, "one tile_start entry per lane");

// The lane's four code bytes of a group that the end of the tensor cuts, in the layout without padding
// (bytes whose first element lies past the end do not exist): byte j = elements 2 (j & 1) + 64 (j >> 1)
// + 4 lane16 and the one after it.
__device__ __forceinline__ uint32_t load_codes_guarded(const uint8_t *codes, int64_t gbase, int lane16, int64_t n)
{
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t e = gbase + lane16 * 4 + (j & 1) * 2 + (j >> 1) * 64;
        if (e < n)
            w |= (uint32_t)codes[e >> 1] << (8 * j);
    }
    return w;
}

__device__ __forceinline__ void store_codes_guarded(uint8_t *codes, int64_t gbase, int lane16, int64_t n, uint32_t w)
{
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t e = gbase + lane16 * 4 + (j & 1) * 2 + (j >> 1) * 64;
        // an element past the end leaves its nibble 0 (lpmm/cpp_extension/fused_adamw_kernel.cu:148-167)
        const uint32_t byte = (w >> (8 * j)) & (e + 1 < n ? 0xFFu : 0x0Fu);
        if (e < n)
            codes[e >> 1] = (uint8_t)byte;
    }
}

// FUSED: the half instantiation of the reference's fused 4-bit operator
// (lpmm/cpp_extension/fused_adamw_kernel.cu:80-174 with T = at::Half) instead of the chain of PyTorch
// ops: codes and scales without padding, the map entry rounded to half before it meets the scale
// ((T)qmap[idx] * scale, a product of halfs), moments and parameter rounded to half where the kernel
// assigns them to T, everything else in float -- the normalised values included.
// USUAL: half_elts8.
template <bool FUSED, bool USUAL>
__global__ __launch_bounds__(kThreads) void adamw4bit_half_kernel(const MultiH args, const Hyper fh,
                                                                 const float *__restrict__ qmap_m,
                                                                 const float *__restrict__ qmap_v)
{
    __shared__ __align__(16) uint32_t lds[(FUSED ? kLdsBytes : kHalfLdsBytes) / 4];
    const int lane = threadIdx.x & (kWave - 1);
    const bool started = lane + 1 < kHMax && args.tile_start[lane + 1] <= blockIdx.x;
    const int lo = __popcll(__ballot(started));
    const TensorH &t = args.t[lo];
    const uint32_t tiles_in_tensor = args.tile_start[lo + 1] - args.tile_start[lo];
    // 4 KB of parameters per tile: 32 tiles make a 128 KB run of an XCD
    const uint32_t tile = xcd_run_order<5>(blockIdx.x - args.tile_start[lo], tiles_in_tensor,
                                           run_phase<5>(t.p, kHTile * sizeof(h16)));
    const int lane16 = threadIdx.x & 15;
    const int64_t n = t.n;
    const int64_t n_groups = (n + kGroup - 1) / kGroup;
    const int64_t grp = (int64_t)tile * (kHTile / kGroup) + (threadIdx.x >> 4);
    const int64_t gbase = grp * kGroup;
    const bool live = grp < n_groups;  // else: a group the padding to whole pack groups added
    const bool full = live && t.vec != 0 && gbase + kGroup <= n;

    h16 *pp = t.p + gbase + lane16 * 4;
    uint16_t *mcp = reinterpret_cast<uint16_t *>(t.mc + (gbase >> 1)) + lane16;
    uint16_t *vcp = reinterpret_cast<uint16_t *>(t.vc + (gbase >> 1)) + lane16;
    LdsFill fill;
    HalfLdsFill half_fill;
    if constexpr (FUSED)
        fill = lds_fill_load(qmap_m, qmap_v);
    else
        half_fill = half_lds_load(qmap_m, qmap_v);
    v2h p2[kPairs], g2[kPairs];
    uint32_t wm = 0, wv = 0;
    float sm = 0.0f, sv = 0.0f;
    if (full) {
        const h16 *gp = t.g + gbase + lane16 * 4;
        const v4h a0 = load_h4(pp), a1 = load_h4(pp + 64), b0 = load_h4(gp), b1 = load_h4(gp + 64);
        pairs_of(a0, a1, p2);
        pairs_of(b0, b1, g2);
    } else if (live) {
#pragma unroll
        for (int k = 0; k < kEltsPerLane; ++k) {
            const int64_t i = gbase + elt_offset(lane16, k);
            p2[k >> 1][k & 1] = i < n ? t.p[i] : (h16)0.0f;
            g2[k >> 1][k & 1] = i < n ? t.g[i] : (h16)0.0f;
        }
    }
    if (live) {
        if (!FUSED || full) {
            // padded to whole pack groups (the chain's layout), or a whole group: always inside
            wm = load_u16(mcp) | (load_u16(mcp + 16) << 16);
            wv = load_u16(vcp) | (load_u16(vcp + 16) << 16);
        } else {
            wm = load_codes_guarded(t.mc, gbase, lane16, n);
            wv = load_codes_guarded(t.vc, gbase, lane16, n);
        }
        sm = (float)t.ms[grp];
        sv = (float)t.vs[grp];
    }
    if constexpr (FUSED)
        lds_fill_store(lds, fill);
    else
        half_lds_store(lds, half_fill);
    const int kind_m = classify_map(qmap_m), kind_v = classify_map(qmap_v);
    lds_barrier();

    if (!FUSED && threadIdx.x == 0 && tile + 1 == tiles_in_tensor) {
        // the tensor's last tile also owns the extra byte at the end of the code buffers
        t.mc[(int64_t)tiles_in_tensor * (kHTile / 2)] = 0;
        t.vc[(int64_t)tiles_in_tensor * (kHTile / 2)] = 0;
    }
    if (FUSED && !live)
        return;
    if (!live) {
        const v2h z[kPairs] = {};
        const uint32_t zm = encode8_half(lds, kLdsQ0, kind_m, z), zv = encode8_half(lds, kLdsQ1, kind_v, z);
        store_u16(mcp, zm & 0xFFFFu);
        store_u16(mcp + 16, zm >> 16);
        store_u16(vcp, zv & 0xFFFFu);
        store_u16(vcp + 16, zv >> 16);
        return;
    }

    NfHyper h;
    h.decay = args.decay;
    h.w1 = args.w1;
    h.b2 = args.b2;
    h.w2 = args.w2;
    h.eps = args.eps;
    h.neg_step_size = t.neg_step_size;
    h.bc2_sqrt = t.bc2_sqrt;
    h.rbc2_sqrt = t.rbc2_sqrt;
    float amax_m = 0.0f, amax_v = 0.0f;
    uint32_t om, ov;
    if constexpr (FUSED) {
        const Nibbles nm = split_nibbles(wm), nv = split_nibbles(wv);
        float m[kEltsPerLane], v[kEltsPerLane];
#pragma unroll
        for (int k = 0; k < kEltsPerLane; ++k) {
            m[k] = rh(rh(decode_nibble(lds, kLdsQ0, nm, k)) * sm);
            v[k] = rh(rh(decode_nibble(lds, kLdsQ1, nv, k)) * sv);
            adamw_moments((float)g2[k >> 1][k & 1], m[k], v[k], fh);
            m[k] = rh(m[k]);
            v[k] = rh(v[k]);
            p2[k >> 1][k & 1] = (h16)rh(adamw_param((float)p2[k >> 1][k & 1], m[k], v[k], fh));
            // elements past the end of the tensor: threads that the operator does not have
            if (!full && gbase + elt_offset(lane16, k) >= n)
                m[k] = v[k] = 0.0f;
            amax_m = fmaxf(amax_m, fabsf(m[k]));
            amax_v = fmaxf(amax_v, fabsf(v[k]));
        }
        row16_max2(amax_m, amax_v);
        // the fused operator normalises in float
        om = encode8_scaled(lds, kLdsQ0, kind_m, m, amax_m);
        ov = encode8_scaled(lds, kLdsQ1, kind_v, v, amax_v);
    } else {
        const MixConst c = mix_const();
        v2h m[kPairs], v[kPairs], scale[kPairs];
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            scale[j] = v2h{(h16)sv, (h16)sv};
        half_decode_m(lds, wm, sm, m);
        half_decode_v(lds, kind_v, wv, scale, v, c);
        half_elts8<false, false, USUAL>(p2, g2, m, v, h, c);
        if (!full) {
            // elements past the end of the tensor: the zero padding of the chain's quantiser
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k)
                if (gbase + elt_offset(lane16, k) >= n)
                    m[k >> 1][k & 1] = v[k >> 1][k & 1] = (h16)0.0f;
        }
        amax_m = max8<true>(m);
        amax_v = max8<false>(v);
        row16_max2(amax_m, amax_v);
        // the chain normalises in half (x.div(max1) on half tensors)
        om = encode8_scaled_h(lds, kLdsQ0, kind_m, m, amax_m, c);
        ov = encode8_scaled_h(lds, kLdsQ1, kind_v, v, amax_v, c);
    }
    if (full) {
        store_pairs(pp, p2);
    } else {
#pragma unroll
        for (int k = 0; k < kEltsPerLane; ++k) {
            const int64_t i = gbase + elt_offset(lane16, k);
            if (i < n)
                t.p[i] = p2[k >> 1][k & 1];
        }
    }
    if (!FUSED || full) {
        store_u16(mcp, om & 0xFFFFu);
        store_u16(mcp + 16, om >> 16);
        store_u16(vcp, ov & 0xFFFFu);
        store_u16(vcp + 16, ov >> 16);
    } else {
        store_codes_guarded(t.mc, gbase, lane16, n, om);
        store_codes_guarded(t.vc, gbase, lane16, n, ov);
    }
    if (lane16 == 0) {
        t.ms[grp] = (h16)amax_m;
        t.vs[grp] = (h16)amax_v;
    }
}

// ---------------------------------------------------------------------------------------
// The chain on float16 states that are not quantised (4096 values or fewer by default), many tensors per
// launch.  As PyTorch ops they are eight to ten launches a tensor: with eight 4096-long norm weights, 80-140 of
// the 1846 us of a step on four decoder layers (1703-1766 now), and most of a small model's step.
// ---------------------------------------------------------------------------------------
constexpr int kHPlainMax = 64;

static_assert(kHTile == kOpsBlock, "a tile is rounded one way");

struct TensorHPlain {
    h16 *p;
    const h16 *g;
    h16 *m, *v;
    int64_t n;
    float neg_step_size, bc2_sqrt;
};

struct MultiHPlain {
    TensorHPlain t[kHPlainMax];
    uint32_t tile_start[kHPlainMax + 1];
    float decay, w1, b2, w2, eps;
};
static_assert(sizeof(MultiHPlain) <= 4096, "kernel arguments exceed 4 KB");

__global__ __launch_bounds__(kThreads) void nonfused_half_plain_kernel(const MultiHPlain args)
{
    const int lane = threadIdx.x & (kWave - 1);
    const bool started = lane + 1 < kHPlainMax && args.tile_start[lane + 1] <= blockIdx.x;
    const int lo = __popcll(__ballot(started));
    const TensorHPlain &t = args.t[lo];
    // a lane's eight values lie 256 apart: coalesced at any alignment
    const int64_t i0 = (int64_t)(blockIdx.x - args.tile_start[lo]) * kHTile + threadIdx.x;
    NfHyper h;
    h.decay = args.decay;
    h.w1 = args.w1;
    h.b2 = args.b2;
    h.w2 = args.w2;
    h.eps = args.eps;
    h.neg_step_size = t.neg_step_size;
    h.bc2_sqrt = t.bc2_sqrt;
    v2h p[kPairs], g[kPairs], m[kPairs], v[kPairs];
#pragma unroll
    for (int k = 0; k < kEltsPerLane; ++k) {
        const int64_t i = i0 + k * kThreads;
        const bool in = i < t.n;
        p[k >> 1][k & 1] = in ? t.p[i] : (h16)0.0f;
        g[k >> 1][k & 1] = in ? t.g[i] : (h16)0.0f;
        m[k >> 1][k & 1] = in ? t.m[i] : (h16)0.0f;
        v[k >> 1][k & 1] = in ? t.v[i] : (h16)0.0f;
    }
    const int64_t tile_end = i0 - threadIdx.x + kHTile;
    const RoundOnce once = {tile_end <= ops_twice(t.v, nullptr, t.n) ? 0u : 0xffu, tile_end <= ops_twice(t.g, t.v, t.n) ? 0u : 0xffu};
    half_elts8<true, true>(p, g, m, v, h, mix_const(), once);
#pragma unroll
    for (int k = 0; k < kEltsPerLane; ++k) {
        const int64_t i = i0 + k * kThreads;
        if (i < t.n) {
            t.p[i] = p[k >> 1][k & 1];
            t.m[i] = m[k >> 1][k & 1];
            t.v[i] = v[k >> 1][k & 1];
        }
    }
}

// ---------------------------------------------------------------------------------------
// Two passes: rank-1 second moment on matrices whose column count is a multiple of 128.  The records
// are MultiR1 with p, g, ms, row_old and col_old pointing at halfs; row_new and col_new are the float
// work arrays.
// ---------------------------------------------------------------------------------------
// Where a lane stands in the operands; a pass moves every pointer on by the same distance, which costs an
// addition each (recomputing them from the row took a tenth of the pass's instructions).
struct HalfCursor {
    h16 *p, *ms;
    const h16 *g, *row_old;
    uint16_t *mc, *vc;
    int64_t row, rows_on, values_on;

    __device__ __forceinline__ HalfCursor(const TensorR1 &t, const Geometry &q, int lane16)
    {
        const int64_t grp = q.row0 * t.col_blocks + q.cg, first = grp * kGroup + lane16 * 4;
        p = reinterpret_cast<h16 *>(t.p) + first;
        g = reinterpret_cast<const h16 *>(t.g) + first;
        ms = reinterpret_cast<h16 *>(t.ms) + grp;
        row_old = reinterpret_cast<const h16 *>(t.row_old) + q.row0;
        mc = reinterpret_cast<uint16_t *>(t.mc) + grp * (kGroup / 4) + lane16;
        vc = reinterpret_cast<uint16_t *>(t.vc) + grp * (kGroup / 4) + lane16;
        row = q.row0;
        rows_on = q.step;
        values_on = (int64_t)q.step * t.col_blocks * kGroup;
    }
    __device__ __forceinline__ void advance()
    {
        p += values_on;
        g += values_on;
        ms += values_on / kGroup;
        row_old += rows_on;
        mc += values_on / 4;
        vc += values_on / 4;
        row += rows_on;
    }
};

// larger of two non-negative floats that are numbers
__device__ __forceinline__ float max_bits(float a, float b)
{
    return __uint_as_float(max(__float_as_uint(a), __float_as_uint(b)));
}

template <bool USUAL>
__global__ __launch_bounds__(kThreads, 6) void rank1_update_half_kernel(const MultiR1 args, const float *__restrict__ qmap_m,
                                                                    const float *__restrict__ qmap_v)
{
    __shared__ __align__(16) uint32_t lds[kHalfLdsBytes / 4];
    __shared__ __align__(16) h16 col_old[kMaxWide * kGroup];
    __shared__ uint32_t colred[kMaxWide * kRedSlotWords];
    __shared__ uint32_t rowred[kRowSlots];
    const int lo = find_tensor(args);
    const TensorR1 &t = args.t[lo];
    const h16 *const COL_OLD = reinterpret_cast<const h16 *>(t.col_old);
    const uint32_t tl = blockIdx.x - args.tile_start[lo];
    const int lane16 = threadIdx.x & 15, drow = threadIdx.x >> 4;
    const Geometry q = geometry(t, tl, drow);
    const int64_t cols = (int64_t)t.col_blocks * kGroup;
    const int64_t tile_c0 = (int64_t)q.col_tile * q.wide * kGroup;
    half_lds_fill(lds, qmap_m, qmap_v);
    for (int j = threadIdx.x; j < kMaxWide * kGroup; j += kThreads)
        col_old[j] = (j < q.wide * kGroup && tile_c0 + j < cols) ? COL_OLD[tile_c0 + j] : (h16)0.0f;
    for (int j = threadIdx.x; j < kMaxWide * (int)kRedSlotWords; j += kThreads)
        colred[j] = 0u;
    if (threadIdx.x < kRowSlots)
        rowred[threadIdx.x] = 0u;
    const int kind_m = classify_map(qmap_m), kind_v = classify_map(qmap_v);
    NfHyper h;
    h.decay = args.decay;
    h.w1 = args.w1;
    h.b2 = args.b2;
    h.w2 = args.w2;
    h.eps = args.eps;
    h.neg_step_size = t.neg_step_size;
    h.bc2_sqrt = t.bc2_sqrt;
    h.rbc2_sqrt = t.rbc2_sqrt;
    const MixConst c = mix_const();
    __syncthreads();

    if (tl == 0) {
        const v2h z[kPairs] = {};
        const int64_t n = t.rows * cols;
        write_padding(t.mc, n, (n + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP,
                      encode8_half(lds, kLdsQ0, kind_m, z));
    }
    const int slot = drow & (q.wide - 1);
    if (q.cg < t.col_blocks && q.row0 < t.rows) {
        const v4h *cop = reinterpret_cast<const v4h *>(col_old + slot * kGroup + lane16 * 4);
        v2h co[kPairs], vtop[kPairs];  // the lane's columns: current statistics, maxima over its passes
        pairs_of(cop[0], cop[16], co);
#pragma unroll
        for (int j = 0; j < kPairs; ++j) {
            co[j] = rank1_columns(co[j]);
            vtop[j] = v2h{(h16)0.0f, (h16)0.0f};
        }
        HalfCursor at(t, q, lane16);
#pragma unroll 1
        for (int it = 0; it < q.passes && at.row < t.rows; ++it, at.advance()) {
            const v4h a0 = load_h4(at.p), a1 = load_h4(at.p + 64), b0 = load_h4(at.g), b1 = load_h4(at.g + 64);
            const uint32_t wm = load_u16(at.mc) | (load_u16(at.mc + 16) << 16);
            const uint32_t wv = load_u16(at.vc) | (load_u16(at.vc + 16) << 16);
            const float sm = (float)*at.ms;
            const h16 ro = *at.row_old;
            v2h p2[kPairs], g2[kPairs], m[kPairs], v[kPairs], s[kPairs];
            pairs_of(a0, a1, p2);
            pairs_of(b0, b1, g2);
#pragma unroll
            for (int j = 0; j < kPairs; ++j)
                s[j] = rank1_scales(co[j], ro);
            half_decode_m(lds, wm, sm, m);
            half_decode_v(lds, kind_v, wv, s, v, c);
            half_elts8<false, false, USUAL>(p2, g2, m, v, h, c);
#pragma unroll
            for (int j = 0; j < kPairs; ++j)
                vtop[j] = max2_bits(vtop[j], v[j]);
            float amax_m = max8<true>(m), vmax = max8<false>(v);
            row16_max2(amax_m, vmax);
            const uint32_t om = encode8_scaled_h(lds, kLdsQ0, kind_m, m, amax_m, c);
            store_pairs(at.p, p2);
            store_u16(at.mc, om & 0xFFFFu);
            store_u16(at.mc + 16, om >> 16);
            if (lane16 == 0) {
                *at.ms = (h16)amax_m;
                atomicMax(rowred + row_slot(t.tile, it, drow), __float_as_uint(vmax));
            }
        }
        uint32_t *red = colred + slot * kRedSlotWords + lane16;
#pragma unroll
        for (int k = 0; k < kEltsPerLane; ++k)
            atomicMax(red + k * 16, __float_as_uint((float)vtop[k >> 1][k & 1]));
    }
    __syncthreads();
    flush_row_maxima(rowred, t.tile, q, drow, t.rows, t.row_new);
    // column j of the tile = element k of lane l of slot s
    for (int j = threadIdx.x; j < q.wide * kGroup; j += kThreads) {
        const int w = j & (kGroup - 1);
        const int k = ((w >> 6) << 2) | (w & 3), l = (w >> 2) & 15;
        if (tile_c0 + j < cols)
            atomic_max_nonneg(t.col_new + tile_c0 + j, __uint_as_float(colred[(j >> 7) * kRedSlotWords + k * 16 + l]));
    }
}

__global__ __launch_bounds__(kThreads, 6) void rank1_requant_half_kernel(const MultiR1 args, const float *__restrict__ qmap_m,
                                                                     const float *__restrict__ qmap_v)
{
    __shared__ __align__(16) uint32_t lds[kHalfLdsBytes / 4];
    __shared__ __align__(16) h16 col_old[kMaxWide * kGroup];
    __shared__ __align__(16) float col_new[kMaxWide * kGroup], col_rcp[kMaxWide * kGroup];
    __shared__ uint32_t odd_columns;  // does the tile have a column statistic outside the reciprocal's exact range
    const int lo = find_tensor(args);
    const TensorR1 &t = args.t[lo];
    const h16 *const COL_OLD = reinterpret_cast<const h16 *>(t.col_old);
    const uint32_t tl = blockIdx.x - args.tile_start[lo];
    const int lane16 = threadIdx.x & 15, drow = threadIdx.x >> 4;
    const Geometry q = geometry(t, tl, drow);
    const int64_t cols = (int64_t)t.col_blocks * kGroup;
    const int64_t tile_c0 = (int64_t)q.col_tile * q.wide * kGroup;
    const int kind_v = classify_map(qmap_v);
    half_lds_fill(lds, qmap_m, qmap_v);
    if (threadIdx.x == 0)
        odd_columns = 0u;
    __syncthreads();
    for (int j = threadIdx.x; j < kMaxWide * kGroup; j += kThreads) {
        const bool in = j < q.wide * kGroup && tile_c0 + j < cols;
        const float cn = in ? t.col_new[tile_c0 + j] : 1.0f;
        col_old[j] = in ? COL_OLD[tile_c0 + j] : (h16)0.0f;
        col_new[j] = cn;
        col_rcp[j] = rcp_exact(cn);
        if (!rc_safe(cn))
            odd_columns = 1u;
    }
    NfHyper h;
    h.b2 = args.b2;
    h.w2 = args.w2;
    const MixConst c = mix_const();
    __syncthreads();

    if (tl == 0) {
        const v2h z[kPairs] = {};
        const int64_t n = t.rows * cols;
        write_padding(t.vc, n, (n + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP,
                      encode8_half(lds, kLdsQ1, kind_v, z));
    }
    if (q.cg >= t.col_blocks)
        return;
    const int col_off = (drow & (q.wide - 1)) * kGroup + lane16 * 4;
    const v4h *cop = reinterpret_cast<const v4h *>(col_old + col_off);
    v2h co[kPairs];
    float rcn[kEltsPerLane];
    pairs_of(cop[0], cop[16], co);
#pragma unroll
    for (int j = 0; j < kPairs; ++j)
        co[j] = rank1_columns(co[j]);
    unpack8(*reinterpret_cast<const float4 *>(col_rcp + col_off), *reinterpret_cast<const float4 *>(col_rcp + col_off + 64), rcn);
    const bool even = kind_v == kMapStdV && __builtin_amdgcn_readfirstlane(odd_columns) == 0u;
    const uint32_t code_dword = code_dword_of_lane(lane16), code_sel = code_swap_selector(lane16);
    const int64_t first = (q.row0 * t.col_blocks + q.cg) * kGroup, values_on = (int64_t)q.step * t.col_blocks * kGroup;
    const h16 *gp = reinterpret_cast<const h16 *>(t.g) + first + lane16 * 4;
    uint32_t *vcp = reinterpret_cast<uint32_t *>(t.vc) + first / 8 + code_dword;
    const h16 *row_old = reinterpret_cast<const h16 *>(t.row_old) + q.row0;
    const float *row_new = t.row_new + q.row0;
    const int64_t rows = t.rows;
#pragma unroll 1
    for (int64_t it = 0, r = q.row0; it < q.passes && r < rows; ++it, r += q.step, gp += values_on, vcp += values_on / 8,
                 row_old += q.step, row_new += q.step) {
        const v4h b0 = load_h4(gp), b1 = load_h4(gp + 64);
        const uint32_t wv = swap_code_halves(load_u32(vcp), code_sel);
        const h16 ro = *row_old;
        const float rn = *row_new;
        v2h g2[kPairs], v[kPairs], s[kPairs], x[kPairs];
        pairs_of(b0, b1, g2);
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            s[j] = rank1_scales(co[j], ro);
        half_decode_v(lds, kind_v, wv, s, v, c);
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            v[j] = half_second_moment(v[j], g2[j], h, c);
        uint32_t ov;
        // every scale is a maximum over the values it divides: where all of the wave's scales lie in the
        // range in which the reciprocal is exact, one product gives the quotient as a half, and the reciprocal
        // of the smaller statistic is the larger of the two reciprocals (rounding is monotonic)
        if (even && __all(rc_safe(rn))) {
            const float rcr = rcp_exact(rn);
#pragma unroll
            for (int j = 0; j < kPairs; ++j)
                x[j] = half_quotients(v[j], max_bits(rcn[2 * j], rcr), max_bits(rcn[2 * j + 1], rcr), c);
            ov = encode8_half_v(x);  // quotients in [0, 1]
        } else {
#pragma unroll
            for (int j = 0; j < kPairs; ++j) {
                v2h pair = v[j];
                asm volatile("" : "+v"(pair));  // what only this branch needs stays in it
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int k = 2 * j + i;
                    const float cn = col_new[col_off + (k & 3) + (k >> 2) * 64];
                    x[j][i] = (h16)rh((float)pair[i] / ((cn < rn) ? cn : rn));
                }
            }
            ov = encode8_half(lds, kLdsQ1, kind_v, x);
        }
        store_u32(vcp, swap_code_halves(ov, code_sel));
    }
}

void launch_rank1_half(const R1Launch &l, const float *qmap_m, const float *qmap_v, hipStream_t stream)
{
    const auto update = half_near(l.update.w1) && half_eps_positive(l.update.eps) ? rank1_update_half_kernel<true> : rank1_update_half_kernel<false>;
    hipLaunchKernelGGL(update, dim3(l.update_tiles), dim3(kThreads), 0, stream, l.update, qmap_m, qmap_v);
    hipLaunchKernelGGL(rank1_requant_half_kernel, dim3(l.requant_tiles), dim3(kThreads), 0, stream, l.requant, qmap_m, qmap_v);
}

// The maxima in the float work arrays, written out as the half statistics of the state.
constexpr int kNarrowMax = 3 * kR1Max;  // arrays per launch (two or three per tensor)

struct NarrowArgs {
    const float *src[kNarrowMax];
    h16 *dst[kNarrowMax];
    int64_t n[kNarrowMax];
};
static_assert(sizeof(NarrowArgs) <= 4096, "kernel arguments exceed 4 KB");

__global__ __launch_bounds__(kThreads) void narrow_stats_kernel(const NarrowArgs args)
{
    const float *src = args.src[blockIdx.y];
    h16 *dst = args.dst[blockIdx.y];
    const int64_t n = args.n[blockIdx.y];
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        dst[i] = (h16)src[i];
}

}  // namespace lpmm

using namespace lpmm;

// FUSED: the operator's arithmetic and layout on one tensor (float hyperparameters, as its signature has them)
template <bool FUSED>
static int half_step_multi(const lpmm_adamw4bit_f16_tensor *tensors, int64_t count, const float *qmap_m,
                           const float *qmap_v, double beta1, double beta2, double lr, double weight_decay, double eps,
                           void *stream)
{
    if (FUSED && count != 1)
        return LPMM_ERR_ARG;
    if (count < 0)
        return LPMM_ERR_SIZE;
    if (count == 0)
        return LPMM_OK;
    LPMM_REQUIRE_PTR(tensors);
    LPMM_REQUIRE_PTR(qmap_m);
    LPMM_REQUIRE_PTR(qmap_v);
    LPMM_REQUIRE_ALIGN(qmap_m, 4);
    LPMM_REQUIRE_ALIGN(qmap_v, 4);
    for (int64_t i = 0; i < count; ++i) {
        const lpmm_adamw4bit_f16_tensor &t = tensors[i];
        if (t.n < 0 || (t.n + kHTile - 1) / kHTile > 0x7fffffffLL)
            return LPMM_ERR_SIZE;
        if (t.n == 0)
            continue;
        LPMM_REQUIRE_PTR(t.p);
        LPMM_REQUIRE_PTR(t.g);
        LPMM_REQUIRE_PTR(t.m_codes);
        LPMM_REQUIRE_PTR(t.m_max1);
        LPMM_REQUIRE_PTR(t.v_codes);
        LPMM_REQUIRE_PTR(t.v_max1);
        LPMM_REQUIRE_ALIGN(t.p, 2);
        LPMM_REQUIRE_ALIGN(t.g, 2);
        LPMM_REQUIRE_ALIGN(t.m_codes, 2);
        LPMM_REQUIRE_ALIGN(t.v_codes, 2);
        LPMM_REQUIRE_ALIGN(t.m_max1, 2);
        LPMM_REQUIRE_ALIGN(t.v_max1, 2);
    }
    const NfHyper c = make_nf_hyper(beta1, beta2, lr, weight_decay, eps, 1.0);
    NfHypers hypers(beta1, beta2, lr, weight_decay, eps);
    MultiH args;
    args.decay = c.decay;
    args.w1 = c.w1;
    args.b2 = c.b2;
    args.w2 = c.w2;
    args.eps = c.eps;
    Hyper fh;
    fh.beta1 = (float)beta1;
    fh.beta2 = (float)beta2;
    fh.omb1 = 1 - fh.beta1;  // formed in float, as the operator does
    fh.omb2 = 1 - fh.beta2;
    fh.lr = (float)lr;
    fh.wd = (float)weight_decay;
    fh.eps = (float)eps;
    // bias corrections as the operator computes them per thread, in float
    bias_corrections(fh.beta1, fh.beta2, FUSED ? tensors[0].step : 1.0f, &fh.c1, &fh.c2s);
    fh.rc2s = 1.0f / fh.c2s;
    int64_t i = 0;
    while (i < count) {
        int k = 0;
        uint64_t tiles = 0;
        args.tile_start[0] = 0;
        while (i < count && k < kHMax) {
            const lpmm_adamw4bit_f16_tensor &t = tensors[i];
            if (t.n == 0) {
                ++i;
                continue;
            }
            const uint64_t nt = (uint64_t)((t.n + kHTile - 1) / kHTile);
            if (tiles + nt > 0x7fffffffULL)
                break;
            TensorH &d = args.t[k];
            d.p = static_cast<h16 *>(t.p);
            d.g = static_cast<const h16 *>(t.g);
            d.mc = t.m_codes;
            d.vc = t.v_codes;
            d.ms = static_cast<h16 *>(t.m_max1);
            d.vs = static_cast<h16 *>(t.v_max1);
            d.n = t.n;
            const NfHyper &h = hypers.at(t.step);
            d.neg_step_size = h.neg_step_size;
            d.bc2_sqrt = h.bc2_sqrt;
            d.rbc2_sqrt = h.rbc2_sqrt;
            d.vec = aligned_to(t.p, 8) && aligned_to(t.g, 8);
            tiles += nt;
            args.tile_start[++k] = (uint32_t)tiles;
            ++i;
        }
        if (k == 0)
            continue;
        for (int j = k + 1; j <= kHMax; ++j)
            args.tile_start[j] = (uint32_t)tiles;
        const auto kernel = !FUSED && half_near(c.w1) && half_eps_positive(c.eps) ? adamw4bit_half_kernel<FUSED, !FUSED>
                                                                                  : adamw4bit_half_kernel<FUSED, false>;
        hipLaunchKernelGGL(kernel, dim3((uint32_t)tiles), dim3(kThreads), 0, (hipStream_t)stream, args, fh, qmap_m, qmap_v);
        const int st = launch_status();
        if (st != LPMM_OK)
            return st;
    }
    return LPMM_OK;
}

extern "C" int lpmm_nonfused_adamw4bit_f16_step_multi(const lpmm_adamw4bit_f16_tensor *tensors, int64_t count,
                                                      const float *qmap_m, const float *qmap_v, double beta1,
                                                      double beta2, double lr, double weight_decay, double eps,
                                                      void *stream)
{
    return half_step_multi<false>(tensors, count, qmap_m, qmap_v, beta1, beta2, lr, weight_decay, eps, stream);
}

extern "C" int lpmm_adamw4bit_f16_step(void *p, const void *g, uint8_t *m_codes, uint8_t *v_codes, void *m_scale,
                                       void *v_scale, const float *qmap_m, const float *qmap_v, int64_t n, float beta1,
                                       float beta2, float lr, float weight_decay, float eps, float step, void *stream)
{
    lpmm_adamw4bit_f16_tensor t;
    t.p = p;
    t.g = g;
    t.m_codes = m_codes;
    t.v_codes = v_codes;
    t.m_max1 = m_scale;
    t.v_max1 = v_scale;
    t.n = n;
    t.step = step;
    t.reserved = 0.0f;
    return half_step_multi<true>(&t, 1, qmap_m, qmap_v, beta1, beta2, lr, weight_decay, eps, stream);
}

extern "C" int lpmm_nonfused_adamw4bit_rank1_f16_step_multi(const lpmm_nonfused_rank1_f16_tensor *tensors, int64_t count,
                                                            const float *qmap_m, const float *qmap_v, double beta1,
                                                            double beta2, double lr, double weight_decay, double eps,
                                                            void *stream)
{
    if (count < 0)
        return LPMM_ERR_SIZE;
    if (count == 0)
        return LPMM_OK;
    LPMM_REQUIRE_PTR(tensors);
    // the float kernels' records, with the work arrays as the next statistics: one launch group at a time
    for (int64_t i = 0; i < count; ++i) {
        const lpmm_nonfused_rank1_f16_tensor &t = tensors[i];
        if (t.rows < 0 || t.cols < 0 || t.cols % kGroup != 0)
            return LPMM_ERR_SIZE;
        if (t.rows == 0 || t.cols == 0)
            continue;
        LPMM_REQUIRE_PTR(t.v_rowmax_next);
        LPMM_REQUIRE_PTR(t.v_colmax_next);
        LPMM_REQUIRE_PTR(t.work);
        LPMM_REQUIRE_ALIGN(t.v_rowmax_next, 2);
        LPMM_REQUIRE_ALIGN(t.v_colmax_next, 2);
        LPMM_REQUIRE_ALIGN(t.work, 16);
        if (t.v_rowmax == t.v_rowmax_next || t.v_colmax == t.v_colmax_next)
            return LPMM_ERR_ARG;
    }
    for (int64_t i0 = 0; i0 < count; i0 += kR1Max) {
        const int k = (int)(count - i0 < kR1Max ? count - i0 : kR1Max);
        lpmm_nonfused_rank1_tensor rec[kR1Max];
        NarrowArgs narrow;
        int arrays = 0;
        int64_t longest = 0;
        for (int j = 0; j < k; ++j) {
            const lpmm_nonfused_rank1_f16_tensor &t = tensors[i0 + j];
            lpmm_nonfused_rank1_tensor &d = rec[j];
            // rows floats, then (from the next multiple of four floats on) cols floats
            float *row_work = t.work, *col_work = t.work == nullptr ? nullptr : t.work + (t.rows + 3) / 4 * 4;
            d.p = static_cast<float *>(t.p);
            d.g = static_cast<const float *>(t.g);
            d.m_codes = t.m_codes;
            d.m_max1 = static_cast<float *>(t.m_max1);
            d.v_codes = t.v_codes;
            d.v_rowmax = static_cast<const float *>(t.v_rowmax);
            d.v_colmax = static_cast<const float *>(t.v_colmax);
            d.v_rowmax_next = row_work;
            d.v_colmax_next = col_work;
            d.rows = t.rows;
            d.cols = t.cols;
            d.step = t.step;
            d.reserved = 0.0f;
            if (t.rows == 0 || t.cols == 0)
                continue;
            narrow.src[arrays] = row_work;
            narrow.dst[arrays] = static_cast<h16 *>(t.v_rowmax_next);
            narrow.n[arrays++] = t.rows;
            narrow.src[arrays] = col_work;
            narrow.dst[arrays] = static_cast<h16 *>(t.v_colmax_next);
            narrow.n[arrays++] = t.cols;
            longest = t.rows > longest ? t.rows : longest;
            longest = t.cols > longest ? t.cols : longest;
        }
        const int st = rank1_step_multi_half(rec, k, qmap_m, qmap_v, beta1, beta2, lr, weight_decay, eps, stream);
        if (st != LPMM_OK)
            return st;
        if (arrays == 0)
            continue;
        int64_t blocks = (longest + kThreads - 1) / kThreads;
        blocks = blocks > 64 ? 64 : blocks;
        hipLaunchKernelGGL(narrow_stats_kernel, dim3((uint32_t)blocks, (uint32_t)arrays), dim3(kThreads), 0,
                           (hipStream_t)stream, narrow);
        const int st2 = launch_status();
        if (st2 != LPMM_OK)
            return st2;
    }
    return LPMM_OK;
}

// Any column count: the work array also holds the maxima of the new first moment's groups, which become the
// scales once the second pass has read the old ones.
int lpmm::rank1_any_half(const lpmm_rank1_any_tensor *tensors, int64_t count, const float *qmap_m, const float *qmap_v,
                         double beta1, double beta2, double lr, double weight_decay, double eps, void *stream)
{
    for (int64_t i = 0; i < count; ++i) {
        const lpmm_rank1_any_tensor &t = tensors[i];
        if (t.rows < 0 || t.cols < 0 || (t.cols != 0 && t.rows > INT64_MAX / t.cols))
            return LPMM_ERR_SIZE;
        if (t.rows == 0 || t.cols == 0)
            continue;
        LPMM_REQUIRE_PTR(t.m_max1_next);
        LPMM_REQUIRE_PTR(t.v_rowmax_next);
        LPMM_REQUIRE_PTR(t.v_colmax_next);
        LPMM_REQUIRE_PTR(t.work);
        LPMM_REQUIRE_ALIGN(t.m_max1_next, 2);
        LPMM_REQUIRE_ALIGN(t.v_rowmax_next, 2);
        LPMM_REQUIRE_ALIGN(t.v_colmax_next, 2);
        LPMM_REQUIRE_ALIGN(t.work, 4);
        if (t.v_rowmax == t.v_rowmax_next || t.v_colmax == t.v_colmax_next || t.m_max1 == t.m_max1_next)
            return LPMM_ERR_ARG;
    }
    for (int64_t i0 = 0; i0 < count; i0 += kR1Max) {
        const int k = (int)(count - i0 < kR1Max ? count - i0 : kR1Max);
        lpmm_rank1_any_tensor rec[kR1Max];
        NarrowArgs narrow;
        int arrays = 0;
        int64_t longest = 0;
        for (int j = 0; j < k; ++j) {
            const lpmm_rank1_any_tensor &t = tensors[i0 + j];
            lpmm_rank1_any_tensor &d = rec[j];
            d = t;
            if (t.rows == 0 || t.cols == 0)
                continue;
            float *row_work = t.work, *col_work = row_work + t.rows, *m_work = col_work + t.cols;
            d.v_rowmax_next = row_work;
            d.v_colmax_next = col_work;
            d.m_max1_next = m_work;
            const float *src[3] = {row_work, col_work, m_work};
            void *dst[3] = {t.v_rowmax_next, t.v_colmax_next, t.m_max1_next};
            const int64_t n[3] = {t.rows, t.cols, (t.rows * t.cols + kGroup - 1) / kGroup};
            for (int a = 0; a < 3; ++a) {
                narrow.src[arrays] = src[a];
                narrow.dst[arrays] = static_cast<h16 *>(dst[a]);
                narrow.n[arrays++] = n[a];
                longest = n[a] > longest ? n[a] : longest;
            }
        }
        const int st = rank1_any_step_multi(rec, k, kAnyHalf, 0, qmap_m, 4, nullptr, qmap_v, 4, nullptr, beta1, beta2, lr,
                                            weight_decay, eps, 3, stream);
        if (st != LPMM_OK)
            return st;
        if (arrays == 0)
            continue;
        int64_t blocks = (longest + kThreads - 1) / kThreads;
        blocks = blocks > 64 ? 64 : blocks;
        hipLaunchKernelGGL(narrow_stats_kernel, dim3((uint32_t)blocks, (uint32_t)arrays), dim3(kThreads), 0,
                           (hipStream_t)stream, narrow);
        const int st2 = launch_status();
        if (st2 != LPMM_OK)
            return st2;
    }
    return LPMM_OK;
}

extern "C" int lpmm_nonfused_update_f16_multi(const lpmm_adamw_fp32_tensor *tensors, int64_t count, double beta1,
                                              double beta2, double lr, double weight_decay, double eps, void *stream)
{
    if (count < 0)
        return LPMM_ERR_SIZE;
    if (count == 0)
        return LPMM_OK;
    LPMM_REQUIRE_PTR(tensors);
    for (int64_t i = 0; i < count; ++i) {
        const lpmm_adamw_fp32_tensor &t = tensors[i];
        if (t.n < 0 || (t.n + kHTile - 1) / kHTile > 0x7fffffffLL)
            return LPMM_ERR_SIZE;
        if (t.n == 0)
            continue;
        LPMM_REQUIRE_PTR(t.p);
        LPMM_REQUIRE_PTR(t.g);
        LPMM_REQUIRE_PTR(t.m);
        LPMM_REQUIRE_PTR(t.v);
        LPMM_REQUIRE_ALIGN(t.p, 2);
        LPMM_REQUIRE_ALIGN(t.g, 2);
        LPMM_REQUIRE_ALIGN(t.m, 2);
        LPMM_REQUIRE_ALIGN(t.v, 2);
    }
    const NfHyper c = make_nf_hyper(beta1, beta2, lr, weight_decay, eps, 1.0);
    NfHypers hypers(beta1, beta2, lr, weight_decay, eps);
    MultiHPlain args;
    args.decay = c.decay;
    args.w1 = c.w1;
    args.b2 = c.b2;
    args.w2 = c.w2;
    args.eps = c.eps;
    int64_t i = 0;
    while (i < count) {
        int k = 0;
        uint64_t tiles = 0;
        args.tile_start[0] = 0;
        while (i < count && k < kHPlainMax) {
            const lpmm_adamw_fp32_tensor &t = tensors[i];
            const uint64_t nt = (uint64_t)((t.n + kHTile - 1) / kHTile);
            if (tiles + nt > 0x7fffffffULL)
                break;
            ++i;
            if (nt == 0)
                continue;
            TensorHPlain &d = args.t[k];
            d.p = reinterpret_cast<h16 *>(t.p);
            d.g = reinterpret_cast<const h16 *>(t.g);
            d.m = reinterpret_cast<h16 *>(t.m);
            d.v = reinterpret_cast<h16 *>(t.v);
            d.n = t.n;
            const NfHyper &h = hypers.at(t.step);
            d.neg_step_size = h.neg_step_size;
            d.bc2_sqrt = h.bc2_sqrt;
            tiles += nt;
            args.tile_start[++k] = (uint32_t)tiles;
        }
        if (k == 0)
            continue;
        for (int j = k + 1; j <= kHPlainMax; ++j)
            args.tile_start[j] = (uint32_t)tiles;
        hipLaunchKernelGGL(nonfused_half_plain_kernel, dim3((uint32_t)tiles), dim3(kThreads), 0, (hipStream_t)stream, args);
        const int st = launch_status();
        if (st != LPMM_OK)
            return st;
    }
    return LPMM_OK;
}
