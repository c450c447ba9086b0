// The two passes of the non-fused AdamW step with a rank-1 second moment for code widths of 5 to 8
// bits.  Tiles, records and statistics as in nonfused_rank1.hip.
#include "lpmm_search.hpp"
#include "rank1_tiles.hpp"

namespace lpmm {

// ---------------------------------------------------------------------------------------
// The same two passes for code widths of 5 to 8 bits (lpmm/configs/default_{5,6,7,8}b.yml): one
// code per byte (lpmm/cpp_extension/quantization_kernel.cu:516-533, :656-669), maps of 2^bits
// entries in LDS, decoded by indexing and encoded as the stand-alone quantisers of these widths
// do it: by the reference's search (:397-427), by one read of the map's code table where the
// caller passes one, or by the closed form of the evenly spaced map (the second moment's in every
// shipped configuration; lpmm_search.hpp).  Same tiles and statistics as above; a lane's eight
// codes are two dwords.  21.06 bytes per parameter cross HBM (p 8, g 4 + 4, m codes 2, v codes
// 1 + 2, scales).  LLaMA-7B-shaped set: 24.2 ms per step with 5 bits, 24.4 ms with 8 (the staged
// path 67.6 ms).  Both passes run within 5 % of the rate of their 4-bit counterparts per byte:
// with the arithmetic taken out, with the table instead of the search and with 8-byte instead of
// 4-byte code accesses they take the same time -- the tile structure sets it, not the codes.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t byte_of(uint32_t w0, uint32_t w1, int k)
{
    return ((k < 4 ? w0 : w1) >> (8 * (k & 3))) & 0xFFu;
}

__device__ __forceinline__ uint32_t pack4(const uint32_t (&c)[kEltsPerLane], int h)
{
    return c[4 * h] | (c[4 * h + 1] << 8) | (c[4 * h + 2] << 16) | (c[4 * h + 3] << 24);
}

// Code `zero` into the padding [n, n_padded) of an array of one code per byte and 0 into the extra
// last byte; one workgroup.  n and n_padded are multiples of 4, the array is 4-byte aligned.
__device__ __forceinline__ void write_padding_bytes(uint8_t *codes, int64_t n, int64_t n_padded, uint32_t zero)
{
    for (int64_t i = n + (int64_t)threadIdx.x * 4; i < n_padded; i += kThreads * 4)
        *reinterpret_cast<uint32_t *>(codes + i) = zero * 0x01010101u;
    if (threadIdx.x == 0)
        codes[n_padded] = 0;
}

// WRAPS: tensors may be rows of several tensor rows (rank1_tiles.hpp: Fold).
template <bool KEEP, bool WRAPS>
__global__ __launch_bounds__(kThreads) void rank1_update_bits_kernel(const MultiR1 args, const float *__restrict__ qmap_m,
                                                                    const float *__restrict__ qmap_v, int bits_m,
                                                                    int bits_v, const uint32_t *__restrict__ table_m)
{
    __shared__ float map_m[256], map_v[256];
    __shared__ SearchLds search_m;
    __shared__ BucketLds bucket_m;
    const uint32_t mode = code_table_mode(code_table_tag(table_m), bits_m);
    __shared__ __align__(16) float col_old[kMaxWide * kGroup];
    __shared__ uint32_t colred[kMaxWide * kRedSlotWords];
    constexpr int kSlots = WRAPS ? kFoldSlots : kRowSlots;
    __shared__ uint32_t rowred[kSlots];
    const int lo = find_tensor(args);
    const TensorR1 &t = args.t[lo];
    const uint32_t tl = blockIdx.x - args.tile_start[lo];
    const int lane16 = threadIdx.x & 15, drow = threadIdx.x >> 4;
    const Fold f = fold_of<WRAPS>(t);
    const Geometry q = geometry(t.tile, f.col_blocks, tl, drow);
    const int64_t cols = (int64_t)f.col_blocks * kGroup;
    const int64_t tile_c0 = (int64_t)q.col_tile * q.wide * kGroup;
    fill_map(map_m, qmap_m, bits_m);
    fill_map(map_v, qmap_v, bits_v);
    if (mode == kCodeTable)
        code_table_store(bucket_m, code_table_load(table_m));
    else if (mode == kCodeSearch)
        fill_search(search_m, qmap_m, bits_m);
    for (int j = threadIdx.x; j < kMaxWide * kGroup; j += kThreads)
        col_old[j] = (j < q.wide * kGroup && tile_c0 + j < cols) ? t.col_old[WRAPS ? fold_col(f, (uint32_t)(tile_c0 + j)) : tile_c0 + j] : 0.0f;
    for (int j = threadIdx.x; j < kMaxWide * (int)kRedSlotWords; j += kThreads)
        colred[j] = 0u;
    for (int j = threadIdx.x; j < kSlots; j += kThreads)
        rowred[j] = 0u;
    NfHyper h;
    h.decay = args.decay;
    h.w1 = args.w1;
    h.b2 = args.b2;
    h.w2 = args.w2;
    h.eps = args.eps;
    h.neg_step_size = t.neg_step_size;
    h.bc2_sqrt = t.bc2_sqrt;
    h.rbc2_sqrt = t.rbc2_sqrt;
    __syncthreads();
    const bool map_even = mode == kCodeEven || (mode == kCodeSearch && map_is_even(search_m));

    if (tl == 0) {
        const int64_t n = (f.values + kGroup - 1) / kGroup * kGroup;
        write_padding_bytes(t.mc, n, (n + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP,
                            code1_by_mode(mode, search_m, bucket_m, bits_m, 0.0f));
    }
    const uint32_t mask_m = (1u << bits_m) - 1u, mask_v = (1u << bits_v) - 1u;
    const int slot = drow & (q.wide - 1);
    if (q.cg < f.col_blocks) {
        const FoldSpan span = WRAPS ? fold_span(f, q.cg) : FoldSpan{0, kGroup};
        const bool second_a = WRAPS && (uint32_t)(4 * lane16) >= span.split, second_b = WRAPS && (uint32_t)(64 + 4 * lane16) >= span.split;
        const uint32_t in_tile = WRAPS ? span.first - fold_span(f, q.col_tile * (uint32_t)q.wide).first : 0u;
        const float least = WRAPS && t.tile.drop_nan ? 0.0f : __builtin_nanf("");  // of a column's values
        const float *cop = col_old + slot * kGroup + lane16 * 4;
        uint32_t *red = colred + slot * kRedSlotWords + lane16;
        float co[kEltsPerLane];
        unpack8(*reinterpret_cast<const float4 *>(cop), *reinterpret_cast<const float4 *>(cop + 64), co);
        // the operands of a pass are requested one pass ahead, so that a wave has two passes' loads in
        // flight (LLaMA-7B-shaped set, 8 bits: 24.9-25.1 -> 24.5-24.6 ms per step)
        struct Fetch {
            float4 a0, a1, b0, b1;
            uint32_t wm0, wm1, wv0, wv1;
            float sm, ro, ro1;  // ro1: of the second tensor row
        };
        auto fetch = [&](int it) {
            Fetch x;
            const int64_t r = q.row0 + it * q.step;
            const int64_t grp = r * f.col_blocks + q.cg;
            const int64_t gbase = grp * kGroup;
            if constexpr (WRAPS) {
                // runs beyond the end read the last one
                const int64_t last = f.values - 4, oa = gbase + lane16 * 4, ob = oa + 64;
                const int64_t a = oa < last ? oa : last, b = ob < last ? ob : last;
                x.a0 = load4(t.p + a);
                x.a1 = load4(t.p + b);
                x.b0 = load4_for<KEEP>(t.g + a);
                x.b1 = load4_for<KEEP>(t.g + b);
                x.wm0 = load_u32(reinterpret_cast<const uint32_t *>(t.mc + a));
                x.wm1 = load_u32(reinterpret_cast<const uint32_t *>(t.mc + b));
                x.wv0 = load_u32_for<KEEP>(reinterpret_cast<const uint32_t *>(t.vc + a));
                x.wv1 = load_u32_for<KEEP>(reinterpret_cast<const uint32_t *>(t.vc + b));
                x.sm = t.ms[a >> 7];
                int64_t r0, r1;
                fold_rows(f, span, r, r0, r1);
                x.ro = t.row_old[r0];
                x.ro1 = t.row_old[r1];
                return x;
            }
            const float *pp = t.p + gbase + lane16 * 4;
            const float *gp = t.g + gbase + lane16 * 4;
            const uint32_t *mcp = reinterpret_cast<const uint32_t *>(t.mc + gbase) + lane16;
            const uint32_t *vcp = reinterpret_cast<const uint32_t *>(t.vc + gbase) + lane16;
            x.a0 = load4(pp);
            x.a1 = load4(pp + 64);
            x.b0 = load4_for<KEEP>(gp);
            x.b1 = load4_for<KEEP>(gp + 64);
            x.wm0 = load_u32(mcp);
            x.wm1 = load_u32(mcp + 16);
            x.wv0 = load_u32_for<KEEP>(vcp);
            x.wv1 = load_u32_for<KEEP>(vcp + 16);
            x.sm = t.ms[grp];
            x.ro = t.row_old[r];
            return x;
        };
        Fetch nxt;
        if (q.row0 < f.rows)
            nxt = fetch(0);
#pragma unroll 1
        for (int it = 0; it < q.passes; ++it) {
            const int64_t r = q.row0 + it * q.step;
            const int64_t grp = r * f.col_blocks + q.cg;
            const int64_t gbase = grp * kGroup;
            if (r >= f.rows || (WRAPS && gbase >= f.values))
                break;
            const bool live_a = !WRAPS || gbase + 4 * lane16 < f.values, live_b = !WRAPS || gbase + 4 * lane16 + 64 < f.values;
            const Fetch cur = nxt;
            if (it + 1 < q.passes && r + q.step < f.rows)
                nxt = fetch(it + 1);
            float *pp = t.p + gbase + lane16 * 4;
            uint32_t *mcp = reinterpret_cast<uint32_t *>(t.mc + gbase) + lane16;
            const float4 a0 = cur.a0, a1 = cur.a1, b0 = cur.b0, b1 = cur.b1;
            const uint32_t wm0 = cur.wm0, wm1 = cur.wm1, wv0 = cur.wv0, wv1 = cur.wv1;
            const float sm = cur.sm, ro_a = second_a ? cur.ro1 : cur.ro, ro_b = second_b ? cur.ro1 : cur.ro;
            float pv[kEltsPerLane], gv[kEltsPerLane], m[kEltsPerLane], v[kEltsPerLane];
            unpack8(a0, a1, pv);
            unpack8(b0, b1, gv);
            float amax_m = 0.0f, vmax = 0.0f, vmax1 = 0.0f;  // vmax1: of the second tensor row
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                const float rk = k >= 4 ? ro_b : ro_a;
                m[k] = map_m[byte_of(wm0, wm1, k) & mask_m] * sm;
                v[k] = map_v[byte_of(wv0, wv1, k) & mask_v] * ((co[k] < rk) ? co[k] : rk);
            }
            if (WRAPS && !live_b) {
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
                if (WRAPS && k >= 4)
                    vmax1 = fmaxf(vmax1, v[k]);
                else
                    vmax = fmaxf(vmax, v[k]);
                atomicMax(red + k * 16, __float_as_uint(WRAPS ? fmaxf(v[k], least) : v[k]));
            }
            if (WRAPS) {
                const float a = vmax, b = vmax1;
                vmax = fmaxf(second_a ? 0.0f : a, second_b ? 0.0f : b);
                vmax1 = row16_max(fmaxf(second_a ? a : 0.0f, second_b ? b : 0.0f));
            }
            row16_max2(amax_m, vmax);
            // |m| <= amax: with the correctly rounded reciprocal one multiply and two fmas give the
            // correctly rounded quotient; maxima outside the reciprocal's exact range (0 included:
            // 0/0 must give NaN) take the plain division
            float xs[kEltsPerLane];
            if (__all(rc_safe(amax_m))) {
                const float rc = rcp_exact(amax_m);
#pragma unroll
                for (int k = 0; k < kEltsPerLane; ++k)
                    xs[k] = div_by_rc(m[k], amax_m, rc);
            } else {
#pragma unroll
                for (int k = 0; k < kEltsPerLane; ++k)
                    xs[k] = m[k] / amax_m;
            }
            uint32_t c[kEltsPerLane];
            codes8_by_mode(mode, search_m, bucket_m, bits_m, map_even, xs, c);
            if (live_a)
                store4(pp, make_float4(pv[0], pv[1], pv[2], pv[3]));
            if (live_b)
                store4(pp + 64, make_float4(pv[4], pv[5], pv[6], pv[7]));
            store_u32(mcp, pack4(c, 0));
            store_u32(mcp + 16, pack4(c, 1));
            if (lane16 == 0) {
                t.ms[grp] = amax_m;
                uint32_t *slot = rowred + row_slot(t.tile, it, drow) * (WRAPS ? 2 : 1) + in_tile;  // rank1_tiles.hpp
                atomicMax(slot, __float_as_uint(vmax));
                if (WRAPS && span.split < (uint32_t)kGroup)
                    atomicMax(slot + 1, __float_as_uint(vmax1));
            }
        }
    }
    __syncthreads();
    if (WRAPS)
        flush_row_maxima_fold(rowred, t.tile, q, drow, f, t.row_new);
    else
        flush_row_maxima(rowred, t.tile, q, drow, t.rows, t.row_new);
    // column j of the tile = element k of lane l of slot s
    for (int j = threadIdx.x; j < q.wide * kGroup; j += kThreads) {
        const int w = j & (kGroup - 1);
        const int k = ((w >> 6) << 2) | (w & 3), l = (w >> 2) & 15;
        if (tile_c0 + j < cols)
            atomic_max_nonneg(t.col_new + (WRAPS ? fold_col(f, (uint32_t)(tile_c0 + j)) : tile_c0 + j),
                              __uint_as_float(colred[(j >> 7) * kRedSlotWords + k * 16 + l]));
    }
}

template <bool WRAPS>
__global__ __launch_bounds__(kThreads) void rank1_requant_bits_kernel(const MultiR1 args, const float *__restrict__ qmap_v,
                                                                     int bits_v, const uint32_t *__restrict__ table_v)
{
    __shared__ float map_v[256];
    __shared__ SearchLds search_v;
    __shared__ BucketLds bucket_v;
    const uint32_t mode = code_table_mode(code_table_tag(table_v), bits_v);
    __shared__ __align__(16) float col_old[kMaxWide * kGroup], col_new[kMaxWide * kGroup];
    const int lo = find_tensor(args);
    const TensorR1 &t = args.t[lo];
    const uint32_t tl = blockIdx.x - args.tile_start[lo];
    const int lane16 = threadIdx.x & 15, drow = threadIdx.x >> 4;
    const Fold f = fold_of<WRAPS>(t);
    const Geometry q = geometry(t.tile, f.col_blocks, tl, drow);
    const int64_t cols = (int64_t)f.col_blocks * kGroup;
    const int64_t tile_c0 = (int64_t)q.col_tile * q.wide * kGroup;
    fill_map(map_v, qmap_v, bits_v);
    if (mode == kCodeTable)
        code_table_store(bucket_v, code_table_load(table_v));
    else if (mode == kCodeSearch)
        fill_search(search_v, qmap_v, bits_v);
    for (int j = threadIdx.x; j < kMaxWide * kGroup; j += kThreads) {
        const bool in = j < q.wide * kGroup && tile_c0 + j < cols;
        const int64_t c = WRAPS ? fold_col(f, (uint32_t)(tile_c0 + j)) : tile_c0 + j;
        col_old[j] = in ? t.col_old[c] : 0.0f;
        col_new[j] = in ? t.col_new[c] : 0.0f;
    }
    NfHyper h;
    h.b2 = args.b2;
    h.w2 = args.w2;
    __syncthreads();
    const bool map_even = mode == kCodeEven || (mode == kCodeSearch && map_is_even(search_v));

    if (tl == 0) {
        const int64_t n = (f.values + kGroup - 1) / kGroup * kGroup;
        write_padding_bytes(t.vc, n, (n + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP,
                            code1_by_mode(mode, search_v, bucket_v, bits_v, 0.0f));
    }
    if (q.cg >= f.col_blocks)
        return;
    const FoldSpan span = WRAPS ? fold_span(f, q.cg) : FoldSpan{0, kGroup};
    const bool second_a = WRAPS && (uint32_t)(4 * lane16) >= span.split, second_b = WRAPS && (uint32_t)(64 + 4 * lane16) >= span.split;
    const uint32_t mask_v = (1u << bits_v) - 1u;
    const int col_off = (drow & (q.wide - 1)) * kGroup + lane16 * 4;
    float co[kEltsPerLane], cn[kEltsPerLane];
    unpack8(*reinterpret_cast<const float4 *>(col_old + col_off), *reinterpret_cast<const float4 *>(col_old + col_off + 64), co);
    unpack8(*reinterpret_cast<const float4 *>(col_new + col_off), *reinterpret_cast<const float4 *>(col_new + col_off + 64), cn);
    // the lane's columns through all passes: the correctly rounded reciprocals of their statistics once
    float rcn[kEltsPerLane];
    bool cols_safe = true;
#pragma unroll
    for (int k = 0; k < kEltsPerLane; ++k) {
        rcn[k] = rcp_exact(cn[k]);
        cols_safe = cols_safe && rc_safe(cn[k]);
    }
#pragma unroll 1
    for (int it = 0; it < q.passes; ++it) {
        const int64_t r = q.row0 + it * q.step;
        const int64_t gbase = (r * f.col_blocks + q.cg) * kGroup;
        if (r >= f.rows || (WRAPS && gbase >= f.values))
            break;
        // runs beyond the end read the last one
        const int64_t oa = gbase + lane16 * 4, ob = oa + 64, last = f.values - 4;
        const float4 b0 = load4(t.g + (WRAPS && oa > last ? last : oa)), b1 = load4(t.g + (WRAPS && ob > last ? last : ob));
        uint32_t *vcp = reinterpret_cast<uint32_t *>(t.vc + gbase) + lane16;
        const uint32_t wv0 = load_u32(vcp), wv1 = load_u32(vcp + 16);
        int64_t r0 = r, r1 = r;
        if (WRAPS)
            fold_rows(f, span, r, r0, r1);
        const float ro = t.row_old[r0], rn = t.row_new[r0], ro1 = WRAPS ? t.row_old[r1] : ro, rn1 = WRAPS ? t.row_new[r1] : rn;
        const float ro_a = second_a ? ro1 : ro, ro_b = second_b ? ro1 : ro, rn_a = second_a ? rn1 : rn, rn_b = second_b ? rn1 : rn;
        float gv[kEltsPerLane], v[kEltsPerLane], x[kEltsPerLane];
        unpack8(b0, b1, gv);
#pragma unroll
        for (int k = 0; k < kEltsPerLane; ++k) {
            const float rk = k >= 4 ? ro_b : ro_a;
            v[k] = map_v[byte_of(wv0, wv1, k) & mask_v] * ((co[k] < rk) ? co[k] : rk);
            nonfused_second_moment(v[k], gv[k], h);
        }
        // every scale is a maximum over the values it divides (v <= scale): where all of the wave's
        // scales lie in the range in which the reciprocal is exact, the correctly rounded reciprocal,
        // one multiply and two fmas give the correctly rounded quotient
        if (__all(cols_safe && rc_safe(rn) && rc_safe(rn1))) {
            const float rcr_a = rcp_exact(rn_a), rcr_b = WRAPS ? rcp_exact(rn_b) : rcr_a;
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                const float rnk = k >= 4 ? rn_b : rn_a;
                const bool by_col = cn[k] < rnk;
                x[k] = div_by_rc(v[k], by_col ? cn[k] : rnk, by_col ? rcn[k] : k >= 4 ? rcr_b : rcr_a);
            }
        } else {
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k) {
                const float rnk = k >= 4 ? rn_b : rn_a;
                x[k] = v[k] / ((cn[k] < rnk) ? cn[k] : rnk);
            }
        }
        if (WRAPS && ob > last) {
#pragma unroll
            for (int k = 0; k < kEltsPerLane; ++k)
                if (k >= 4 || oa > last)
                    x[k] = 0.0f;
        }
        uint32_t c[kEltsPerLane];
        codes8_by_mode(mode, search_v, bucket_v, bits_v, map_even, x, c);
        store_u32(vcp, pack4(c, 0));
        store_u32(vcp + 16, pack4(c, 1));
    }
}

void launch_rank1_bits(const R1Launch &l, bool wraps, const float *qmap_m, const float *qmap_v, int bits_m,
                       int bits_v, const uint32_t *table_m, const uint32_t *table_v, hipStream_t stream)
{
    const auto update = wraps ? (l.keep ? rank1_update_bits_kernel<true, true> : rank1_update_bits_kernel<false, true>)
                              : (l.keep ? rank1_update_bits_kernel<true, false> : rank1_update_bits_kernel<false, false>);
    const auto requant = wraps ? rank1_requant_bits_kernel<true> : rank1_requant_bits_kernel<false>;
    hipLaunchKernelGGL(update, dim3(l.update_tiles), dim3(kThreads), 0, stream, l.update, qmap_m, qmap_v, bits_m, bits_v, table_m);
    hipLaunchKernelGGL(requant, dim3(l.requant_tiles), dim3(kThreads), 0, stream, l.requant, qmap_v, bits_v, table_v);
}

}  // namespace lpmm
