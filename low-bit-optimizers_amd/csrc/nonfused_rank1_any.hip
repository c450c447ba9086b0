// The two passes of the non-fused AdamW step with a rank-1 second moment for any column count and any
// alignment, for every kind of state and parameter the tuned kernels serve: 4-bit states (what
// nonfused_rank1_ragged.hip leaves: columns that are no multiple of 8), an fp32 first moment, 5-8-bit
// codes and float16 parameters on columns that are no multiple of 128, operands off a 16-byte boundary.  Tiles, records and statistics
// as in nonfused_rank1.hip.
//
// What the tuned kernels rely on and these do not: rows that start on a 16-byte boundary and on a whole
// code byte, and 128-value groups of the first moment that never straddle a row.  Here
//   * a lane takes columns 16 apart (column block start + 16 k + lane), one value per access, so that
//     neighbouring lanes touch neighbouring addresses whatever the row's first address is;
//   * lanes beyond the end of the row work on the row's last value once more and store nothing: their
//     maxima change nothing, and no access needs a branch;
//   * the first moment's groups lie in up to two pieces in a DPP row's 128 values; its scale takes the
//     route of the second moment's statistics (maxima merged by the first pass, codes written by the
//     second), as in the ragged kernels;
//   * the new codes go to arrays of their own, as on the staged path (the state's tensors are replaced); two codes
//     that share a byte may belong to neighbouring lanes (they meet by a lane exchange) or, where the column
//     count is odd, to different rows: the first pass clears the word around such a byte, the second sets the word's codes
//     by atomic or (store_nibbles).
// Two forms (rank1_any_runs): runs of four neighbouring values a lane where every tensor of a launch allows it, single values 16 apart
// otherwise.  A step on six tensors, single values -> runs (with the order of xcd_neighbours, quotients by reciprocals kept over
// a lane's rows and no load behind a branch): 4096 x 4100 600 -> 486 us, fp32 first moment 620 -> 518, 8 bits 618 -> 540,
// float16 724 -> 528; 4096 x 1600 258 -> 201 (fp32), 264 -> 214 (8 bits), 350 -> 257 (float16).
// Before, these tensors took the staged path (dequantise, update, statistics, normalise: six to eight
// launches a tensor and 50 bytes a value; float16: about thirty PyTorch ops a tensor).  One step on one tensor,
// staged -> here: 4096 x 4100 default 224 -> 107 us, fp32 first moment 183 -> 104, 8 bits 221 -> 102, float16
// 539 -> 151; 4095 x 4099 271 -> 142; 50000 x 34 122 -> 55 (4096 x 4096 on the tuned kernels: 74-84, float16 67).
// What bounds them: instructions; with single values also the code bytes' extraction and one access per value (runs and the tuned
// kernels move the same bytes in a quarter of the accesses); most of the gain on small tensors is launches.
#include "lpmm_half.hpp"
#include "lpmm_search.hpp"

namespace lpmm {

constexpr int kAnyElts = kEltsPerLane;

template <int CTRL>
__device__ __forceinline__ uint32_t any_dpp(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}

__device__ __forceinline__ uint32_t row16_or(uint32_t v)
{
    v |= any_dpp<0xB1>(v);
    v |= any_dpp<0x4E>(v);
    v |= any_dpp<0x141>(v);
    v |= any_dpp<0x140>(v);
    return v;
}

// largest of the DPP row's bit patterns, in every lane
__device__ __forceinline__ uint32_t row16_umax(uint32_t v)
{
    v = max(v, any_dpp<0xB1>(v));   // quad_perm:[1,0,3,2]
    v = max(v, any_dpp<0x4E>(v));   // quad_perm:[2,3,0,1]
    v = max(v, any_dpp<0x141>(v));  // row_half_mirror
    v = max(v, any_dpp<0x140>(v));  // row_mirror
    return v;
}

__device__ __forceinline__ uint32_t magnitude(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// Larger of a maximum so far and |x|, as a bit pattern.  float: a NaN is left out, as by the quantisers' statistics
// (one NaN gradient costs its own parameter and not its row); HALF: it is the maximum, as in the chain of half ops.
template <bool HALF>
__device__ __forceinline__ uint32_t larger(uint32_t top, float x)
{
    return HALF ? max(top, magnitude(x)) : __float_as_uint(fmaxf(__uint_as_float(top), fabsf(x)));
}

// A DPP row's piece of one tensor row: `count` values (1 .. 128) from flattened index `base` on; the values
// from `split` on belong to the next group of the first moment.
struct Piece {
    int64_t base, group;
    int count, split;
};

__device__ __forceinline__ Piece piece_of(int64_t cols, uint32_t cg, int64_t r, int lg_group)
{
    Piece w;
    const int64_t c0 = (int64_t)cg * kGroup;
    w.base = r * cols + c0;
    w.count = (int)(cols - c0 < kGroup ? cols - c0 : kGroup);
    w.group = w.base >> lg_group;
    const int64_t to_next = ((w.group + 1) << lg_group) - w.base;
    w.split = to_next < kGroup ? (int)to_next : kGroup;
    return w;
}

// Which of a piece's values a lane has.  VEC: two runs of four neighbours, 64 apart, as in the tuned kernels (rows of a multiple of four
// values, operands on the boundaries that whole runs need); otherwise values 16 apart.  A lane beyond the piece's end has
// the last run or value once more.
template <bool VEC>
__device__ __forceinline__ bool piece_has(const Piece &w, int lane16, int k)
{
    return (VEC ? 4 * lane16 + 64 * (k >> 2) : 16 * k + lane16) < w.count;
}

template <bool VEC>
__device__ __forceinline__ int piece_at(const Piece &w, int lane16, int k)
{
    const int off = VEC ? 4 * lane16 + 64 * (k >> 2) : 16 * k + lane16;
    return VEC ? (off < w.count ? off : w.count - 4) + (k & 3) : off < w.count ? off : w.count - 1;
}

// KEEP: without the nontemporal hint.  Where rows do not start on cache lines, a line at the edge of a piece is read by two workgroups, and
// the update pass finds it in the L2 the second time (neighbouring tiles are on one XCD: xcd_neighbours).  Six tensors of 4096 x 4100, update
// pass with and without the hint: 294 and 261 us, fp32 first moment 445 and 367, 8 bits 331 and 286; of 4096 x 1600, where rows start on
// lines, fp32 first moment 137 and 139-158.  The second pass reads g for the last time: 125 with the hint, 156 without (fp32).
template <bool KEEP>
__device__ __forceinline__ void load_run(const float *at, float *o)
{
    const float4 a = KEEP ? *reinterpret_cast<const float4 *>(at) : load4(at);
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
}
template <bool KEEP>
__device__ __forceinline__ void load_run(const h16 *at, h16 *o)
{
    const v4h a = KEEP ? *reinterpret_cast<const v4h *>(at) : load_h4(at);
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
}
__device__ __forceinline__ void store_run(float *at, const float *x) { store4(at, make_float4(x[0], x[1], x[2], x[3])); }
__device__ __forceinline__ void store_run(h16 *at, const h16 *x)
{
    __builtin_nontemporal_store(v4h{x[0], x[1], x[2], x[3]}, reinterpret_cast<v4h *>(at));
}

template <bool VEC, bool KEEP, typename T>
__device__ __forceinline__ void load_values(const T *at, const Piece &w, int lane16, T (&o)[kAnyElts])
{
    if constexpr (VEC) {
        load_run<KEEP>(at + piece_at<true>(w, lane16, 0), o);
        load_run<KEEP>(at + piece_at<true>(w, lane16, 4), o + 4);
    } else {
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k)
            o[k] = at[piece_at<false>(w, lane16, k)];
    }
}

template <bool VEC, typename T>
__device__ __forceinline__ void store_values(T *at, const Piece &w, int lane16, const T (&x)[kAnyElts])
{
    if constexpr (VEC) {
        if (piece_has<true>(w, lane16, 0))
            store_run(at + 4 * lane16, x);
        if (piece_has<true>(w, lane16, 4))
            store_run(at + 4 * lane16 + 64, x + 4);
    } else {
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k)
            if (piece_has<false>(w, lane16, k))
                at[16 * k + lane16] = x[k];
    }
}

// The chain of ops has its second moment in a tensor of its own, on a 16-byte boundary; the gradient may lie anywhere.
template <bool VEC>
__device__ __forceinline__ RoundOnce rounded_once(const Piece &w, int lane16, int64_t n, const void *g)
{
    const int64_t twice = ops_twice(nullptr, nullptr, n);
    uint32_t behind = 0;
    if (w.base + w.count > twice)
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k)
            behind |= (w.base + piece_at<VEC>(w, lane16, k) >= twice ? 1u : 0u) << k;
    return RoundOnce{behind, ops_twice(g, nullptr, n) == twice ? behind : 0xffu};
}

// codes of the lane's eight values: element k in bits 4 k (two codes a byte) or in byte k (one a byte)
template <bool BITS, bool VEC>
__device__ __forceinline__ uint64_t load_codes(const uint8_t *codes, const Piece &w, int lane16)
{
    uint64_t out = 0;
    if (VEC) {
        const int64_t a = w.base + piece_at<true>(w, lane16, 0), b = w.base + piece_at<true>(w, lane16, 4);
        if (BITS)
            return load_u32(reinterpret_cast<const uint32_t *>(codes + a)) |
                   (uint64_t)load_u32(reinterpret_cast<const uint32_t *>(codes + b)) << 32;
        return load_u16(reinterpret_cast<const uint16_t *>(codes + (a >> 1))) |
               load_u16(reinterpret_cast<const uint16_t *>(codes + (b >> 1))) << 16;
    }
    if (BITS) {
        const uint8_t *c = codes + w.base;
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k)
            out |= (uint64_t)c[piece_at<false>(w, lane16, k)] << (8 * k);
    } else {
        const uint8_t *c = codes + (w.base >> 1);
        const int odd = (int)(w.base & 1);
        uint32_t low = 0;
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k) {
            const int at = piece_at<false>(w, lane16, k) + odd;
            low |= (((uint32_t)c[at >> 1] >> (4 * (at & 1))) & 15u) << (4 * k);
        }
        out = low;
    }
    return out;
}

// Two codes share a byte, and where the column count is odd the two may belong to different rows, which different
// workgroups write.  An atomic or covers four bytes, so it is the whole word around such a byte that is put together
// this way: in an odd matrix the first pass clears every word that a piece does not fill by itself, the second sets
// the piece's codes of either such word with one atomic, and plain byte stores go only to words that lie wholly
// inside one piece.  No byte is written both ways, and no word by stores of one size while another workgroup
// writes it with the other.  (An atomic per shared byte beside plain stores into the same words took 155 us for
// 4095 x 4099, this 142.)
__device__ __forceinline__ uint32_t *word_of(uint8_t *codes, int64_t flat) { return reinterpret_cast<uint32_t *>(codes) + (flat >> 3); }

// the words that a piece of an odd matrix shares with its neighbours
__device__ __forceinline__ void clear_shared(uint8_t *codes, const Piece &w)
{
    const int64_t end = w.base + w.count;
    if (w.base & 7)
        *word_of(codes, w.base) = 0u;
    if (end & 7)
        *word_of(codes, end) = 0u;
}

__device__ __forceinline__ void store_nibbles(uint8_t *codes, const Piece &w, int lane16, uint32_t now, bool odd_cols)
{
    uint8_t *c = codes + (w.base >> 1);
    const int odd = (int)(w.base & 1);
    const bool low = ((lane16 + odd) & 1) == 0;  // the lane's codes are low halves of their bytes
    // the piece's values in words of its own; an even matrix has no shared bytes
    const int first = odd_cols ? (int)(-w.base & 7) : 0, end = odd_cols ? w.count - (int)((w.base + w.count) & 7) : w.count;
    // the codes one column on: lane 15's are lane 0's of the next sixteen columns
    const int lane = threadIdx.x & (kWave - 1);
    uint32_t next = (uint32_t)__shfl((int)now, (lane & ~15) | ((lane + 1) & 15), kWave);
    if (lane16 == 15)
        next >>= 4;
    if (low) {
        uint8_t *at = c + ((lane16 + odd) >> 1);
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k) {
            const int off = 16 * k + lane16;
            if (off >= first && off < end)
                at[8 * k] = (uint8_t)(((now >> (4 * k)) & 15u) | (((next >> (4 * k)) & 15u) << 4));
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!odd_cols)
        return;
    // at most seven values at either end: a lane has at most its first one there and its last one here
    const int k = (w.count - 1 - lane16) >> 4, off = 16 * k + lane16;
    const uint32_t head = lane16 < first && lane16 < w.count ? (now & 15u) << (4 * ((int)(w.base + lane16) & 7)) : 0u;
    const uint32_t tail = off >= end && off >= first ? ((now >> (4 * (k & 7))) & 15u) << (4 * ((int)(w.base + off) & 7)) : 0u;
    const uint32_t heads = row16_or(head), tails = row16_or(tail);
    if (lane16 == 0) {
        if (heads != 0u)
            atomicOr(word_of(codes, w.base), heads);
        if (tails != 0u)
            atomicOr(word_of(codes, w.base + w.count - 1), tails);
    }
}

// VEC: no two rows share a byte
__device__ __forceinline__ void store_nibble_runs(uint8_t *codes, const Piece &w, int lane16, uint32_t now)
{
    uint16_t *c = reinterpret_cast<uint16_t *>(codes + (w.base >> 1)) + lane16;
    if (piece_has<true>(w, lane16, 0))
        store_u16(c, now & 0xFFFFu);
    if (piece_has<true>(w, lane16, 4))
        store_u16(c + 16, now >> 16);
}

template <bool VEC>
__device__ __forceinline__ void store_bytes(uint8_t *codes, const Piece &w, int lane16, const uint32_t (&now)[kAnyElts])
{
    uint8_t *c = codes + w.base;
    if (VEC) {
        uint32_t *at = reinterpret_cast<uint32_t *>(c) + lane16;
        if (piece_has<true>(w, lane16, 0))
            store_u32(at, now[0] | (now[1] << 8) | (now[2] << 16) | (now[3] << 24));
        if (piece_has<true>(w, lane16, 4))
            store_u32(at + 16, now[4] | (now[5] << 8) | (now[6] << 16) | (now[7] << 24));
        return;
    }
#pragma unroll
    for (int k = 0; k < kAnyElts; ++k) {
        const int off = 16 * k + lane16;
        if (off < w.count)
            c[off] = (uint8_t)now[k];
    }
}

// The codes behind the tensor's n values: `last` up to n_group (the zeros that complete a group are divided by
// its scale like its other values), `zero` up to whole pack groups, 0 in the extra byte.  One workgroup.
template <bool BITS>
__device__ __forceinline__ void any_padding(uint8_t *codes, int64_t n, int64_t n_group, uint32_t last, uint32_t zero, bool odd_cols)
{
    const int64_t n_all = (n_group + LPMM_PACK_GROUP - 1) / LPMM_PACK_GROUP * LPMM_PACK_GROUP;
    if (BITS) {
        for (int64_t i = n + threadIdx.x; i < n_all; i += kThreads)
            codes[i] = (uint8_t)(i < n_group ? last : zero);
        if (threadIdx.x == 0)
            codes[n_all] = 0;
        return;
    }
    // the rest of the last value's word goes the word's way
    const int64_t from = odd_cols ? (n + 7) & ~(int64_t)7 : n;
    if (n + threadIdx.x < from)
        atomicOr(word_of(codes, n), (n + threadIdx.x < n_group ? last : zero) << (4 * ((int)(n + threadIdx.x) & 7)));
    for (int64_t i = from / 2 + threadIdx.x; i < n_all / 2; i += kThreads)
        codes[i] = (uint8_t)((2 * i < n_group ? last : zero) * 0x11u);
    if (threadIdx.x == 0)
        codes[n_all / 2] = 0;
}

// a code array's map: 2^bits floats
template <bool BITS>
__device__ __forceinline__ float any_decode(const float *map, uint64_t codes, int k, uint32_t mask)
{
    return map[BITS ? (uint32_t)(codes >> (8 * k)) & mask : (uint32_t)(codes >> (4 * k)) & 15u];
}

__device__ __forceinline__ float rank1_scale(float co, float ro) { return co < ro ? co : ro; }

// REAL: the parameters' type (h16: the chain of half ops, half scales and statistics, float work arrays for the
// maxima); M32: fp32 first moment; BITS: one code of bits_m / bits_v bits per byte
template <typename REAL, bool M32, bool BITS, bool VEC>
__global__ __launch_bounds__(kThreads, 4) void rank1_update_any_kernel(const MultiR1 args, const NewCodes out,
                                                                       const float *__restrict__ qmap_m,
                                                                       const float *__restrict__ qmap_v, int bits_m, int bits_v)
{
    constexpr bool HALF = sizeof(REAL) == 2;
    constexpr int kMap = BITS ? 256 : 16;
    __shared__ float map_m[kMap], map_v[kMap];
    __shared__ uint32_t colred[kMaxWide * kGroup], rowred[kRowSlots];
    const int lo = find_tensor(args);
    const TensorR1 &t = args.t[lo];
    const uint32_t tl = xcd_neighbours(blockIdx.x - args.tile_start[lo], args.tile_start[lo + 1] - args.tile_start[lo]);
    const int lane16 = threadIdx.x & 15, drow = threadIdx.x >> 4;
    const Geometry q = geometry(t, tl, drow);
    const int64_t cols = (int64_t)(t.col_blocks - 1) * kGroup + t.col_tail;
    fill_map(map_m, qmap_m, BITS ? bits_m : 4);
    fill_map(map_v, qmap_v, BITS ? bits_v : 4);
    for (int j = threadIdx.x; j < kMaxWide * kGroup; j += kThreads)
        colred[j] = 0u;
    if (threadIdx.x < kRowSlots)
        rowred[threadIdx.x] = 0u;
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

    const uint32_t mask_m = (1u << bits_m) - 1u, mask_v = (1u << bits_v) - 1u;
    const int lg_group = 7 + (int)t.m_lg;
    const bool keep = cols % (128 / (int)sizeof(REAL)) != 0;
    if (q.cg < t.col_blocks && q.row0 < t.rows) {
        const REAL *row_old = reinterpret_cast<const REAL *>(t.row_old);
        const REAL *col_old = reinterpret_cast<const REAL *>(t.col_old) + (int64_t)q.cg * kGroup;
        const REAL *ms = reinterpret_cast<const REAL *>(t.ms);
        const Piece first = piece_of(cols, q.cg, q.row0, lg_group);
        REAL co[kAnyElts];
        uint32_t vtop[kAnyElts];  // the lane's columns: current statistics, maxima over its passes
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k) {
            co[k] = col_old[piece_at<VEC>(first, lane16, k)];
            vtop[k] = 0u;
        }
#pragma unroll 1
        for (int it = 0; it < q.passes; ++it) {
            const int64_t r = q.row0 + (int64_t)it * q.step;
            if (r >= t.rows)
                break;
            const Piece w = piece_of(cols, q.cg, r, lg_group);
            REAL *pp = reinterpret_cast<REAL *>(t.p) + w.base;
            const REAL *gp = reinterpret_cast<const REAL *>(t.g) + w.base;
            float *mp = reinterpret_cast<float *>(t.mc) + w.base;
            REAL p[kAnyElts], g[kAnyElts];
            float m[kAnyElts], v[kAnyElts];
            // The small loads: ahead of the branch between the values' loads where a lane takes runs (behind it the compiler
            // waits for values before it issues them), behind single values' loads, where ahead they cost more than they
            // save (72M values in rows of 1682, 4 bits: update 227 -> 206 us with them behind, and the requantisation
            // with the conditional second scale 243 -> 213 us).
            uint64_t vc = 0, mc = 0;
            REAL ro;
            float s0 = 0.0f, s1 = 0.0f;
            const auto small_loads = [&] {
                vc = load_codes<BITS, VEC>(t.vc, w, lane16);
                ro = row_old[r];
                if (!M32) {
                    mc = load_codes<BITS, VEC>(t.mc, w, lane16);
                    s0 = (float)ms[w.group];
                    if (VEC)
                        s1 = (float)ms[w.group + (w.split < w.count ? 1 : 0)];
                    else
                        s1 = w.split < w.count ? (float)ms[w.group + 1] : 0.0f;
                }
            };
            if (VEC)
                small_loads();
            if (keep) {
                load_values<VEC, true>(pp, w, lane16, p);
                load_values<VEC, true>(gp, w, lane16, g);
                if (M32)
                    load_values<VEC, true>(mp, w, lane16, m);
            } else {
                load_values<VEC, false>(pp, w, lane16, p);
                load_values<VEC, false>(gp, w, lane16, g);
                if (M32)
                    load_values<VEC, false>(mp, w, lane16, m);
            }
            if (!VEC)
                small_loads();
            if (!M32) {
#pragma unroll
                for (int k = 0; k < kAnyElts; ++k)
                    m[k] = any_decode<BITS>(map_m, mc, k, mask_m) * (piece_at<VEC>(w, lane16, k) < w.split ? s0 : s1);
            }
#pragma unroll
            for (int k = 0; k < kAnyElts; ++k)
                v[k] = any_decode<BITS>(map_v, vc, k, mask_v) * rank1_scale((float)co[k], (float)ro);
            if constexpr (HALF) {
                const MixConst c = mix_const();
                v2h p2[kPairs], g2[kPairs], m2[kPairs], v2[kPairs];
#pragma unroll
                for (int j = 0; j < kPairs; ++j) {
                    p2[j] = v2h{p[2 * j], p[2 * j + 1]};
                    g2[j] = v2h{g[2 * j], g[2 * j + 1]};
                    m2[j] = round2(m[2 * j], m[2 * j + 1]);
                    v2[j] = round2(v[2 * j], v[2 * j + 1]);
                }
                half_elts8<true, true>(p2, g2, m2, v2, h, c, rounded_once<VEC>(w, lane16, t.rows * cols, t.g));
#pragma unroll
                for (int k = 0; k < kAnyElts; ++k) {
                    p[k] = p2[k >> 1][k & 1];
                    m[k] = (float)m2[k >> 1][k & 1];
                    v[k] = (float)v2[k >> 1][k & 1];
                }
            } else {
#pragma unroll
                for (int k = 0; k < kAnyElts; ++k)
                    nonfused_elt(p[k], g[k], m[k], v[k], h);
            }
            uint32_t vmax = 0u;
#pragma unroll
            for (int k = 0; k < kAnyElts; ++k) {
                vtop[k] = larger<HALF>(vtop[k], v[k]);
                vmax = larger<HALF>(vmax, v[k]);
            }
            vmax = row16_umax(vmax);
            if (!M32) {
                uint32_t m0 = 0u, m1 = 0u;
#pragma unroll
                for (int k = 0; k < kAnyElts; ++k) {
                    const bool here = piece_at<VEC>(w, lane16, k) < w.split;
                    m0 = larger<HALF>(m0, here ? m[k] : 0.0f);
                    m1 = larger<HALF>(m1, here ? 0.0f : m[k]);
                }
                m0 = row16_umax(m0);
                m1 = row16_umax(m1);
                if (lane16 == 0) {
                    // zero changes nothing: the next scales start there
                    if (m0 != 0u)
                        atomic_max_nonneg(t.ms_new + w.group, __uint_as_float(m0));
                    if (m1 != 0u)
                        atomic_max_nonneg(t.ms_new + w.group + 1, __uint_as_float(m1));
                }
            }
            if (lane16 == 0) {
                atomicMax(rowred + row_slot(t.tile, it, drow), vmax);
                if (!BITS && (cols & 1) != 0) {
                    clear_shared(out.v[lo], w);
                    if (!M32)
                        clear_shared(out.m[lo], w);
                }
            }
            store_values<VEC>(pp, w, lane16, p);
            if (M32)
                store_values<VEC>(mp, w, lane16, m);
        }
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k)
            atomicMax(colred + (drow & (q.wide - 1)) * kGroup + piece_at<VEC>(first, lane16, k), vtop[k]);
    }
    __syncthreads();
    flush_row_maxima(rowred, t.tile, q, drow, t.rows, t.row_new);
    const int64_t tile_c0 = (int64_t)q.col_tile * q.wide * kGroup;
    for (int j = threadIdx.x; j < q.wide * kGroup; j += kThreads)
        if (tile_c0 + j < cols)
            atomic_max_nonneg(t.col_new + tile_c0 + j, __uint_as_float(colred[j]));
}

template <bool BITS>
struct AnyCoder;

// 4-bit codes: both maps and the encode table in one LDS array
template <>
struct AnyCoder<false> {
    struct Lds {
        __align__(16) uint32_t w[kLdsBytes / 4];
    };
    Lds &l;
    int kind[2];

    __device__ __forceinline__ AnyCoder(Lds &lds, const float *qm, const float *qv, int, int, const uint32_t *, const uint32_t *) : l(lds)
    {
        lds_fill(l.w, qm, qv);
        kind[0] = classify_map(qm);
        kind[1] = classify_map(qv);
    }
    __device__ __forceinline__ void ready() {}
    __device__ __forceinline__ const float *map(int which) const { return reinterpret_cast<const float *>(l.w) + 16 * which; }
    __device__ __forceinline__ uint32_t one(int which, float x) const
    {
        const float xs[kAnyElts] = {x, x, x, x, x, x, x, x};
        return encode8_plain(l.w, which ? kLdsQ1 : kLdsQ0, kind[which], xs) & 15u;
    }
    template <bool VEC>
    __device__ __forceinline__ void store(int which, const float (&x)[kAnyElts], uint8_t *codes, const Piece &w, int lane16, bool odd_cols) const
    {
        const uint32_t now = encode8_plain(l.w, which ? kLdsQ1 : kLdsQ0, kind[which], x);
        if (VEC)
            store_nibble_runs(codes, w, lane16, now);
        else
            store_nibbles(codes, w, lane16, now, odd_cols);
    }
};

template <>
struct AnyCoder<true> {
    struct Lds {
        float map[2][256];
        SearchLds search[2];
        BucketLds bucket[2];
    };
    Lds &l;
    int bits[2];
    uint32_t mode[2];
    bool even[2];

    __device__ __forceinline__ AnyCoder(Lds &lds, const float *qm, const float *qv, int bm, int bv, const uint32_t *tm, const uint32_t *tv) : l(lds)
    {
        const float *q[2] = {qm, qv};
        const uint32_t *table[2] = {tm, tv};
        bits[0] = bm;
        bits[1] = bv;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            mode[i] = code_table_mode(code_table_tag(table[i]), bits[i]);
            fill_map(l.map[i], q[i], bits[i]);
            if (mode[i] == kCodeTable)
                code_table_store(l.bucket[i], code_table_load(table[i]));
            else if (mode[i] == kCodeSearch)
                fill_search(l.search[i], q[i], bits[i]);
        }
    }
    // after the barrier that follows the constructor
    __device__ __forceinline__ void ready()
    {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            even[i] = mode[i] == kCodeEven || (mode[i] == kCodeSearch && map_is_even(l.search[i]));
    }
    __device__ __forceinline__ const float *map(int which) const { return l.map[which]; }
    __device__ __forceinline__ uint32_t one(int which, float x) const
    {
        return code1_by_mode(mode[which], l.search[which], l.bucket[which], bits[which], x);
    }
    template <bool VEC>
    __device__ __forceinline__ void store(int which, const float (&x)[kAnyElts], uint8_t *codes, const Piece &w, int lane16, bool) const
    {
        uint32_t c[kAnyElts];
        codes8_by_mode(mode[which], l.search[which], l.bucket[which], bits[which], even[which], x, c);
        store_bytes<VEC>(codes, w, lane16, c);
    }
};

// A wave's reciprocals of the scales s[k], and whether they may be used (any_quotients).  KEPT: the caller has them already, from
// statistics that stay over a lane's rows; where a lane takes single values the registers for that are not there (float16, 4095 x 4099:
// 795 -> 982 us a step on six tensors).
template <bool KEPT>
__device__ __forceinline__ bool any_reciprocals(const float (&s)[kAnyElts], float (&rc)[kAnyElts], bool safe)
{
    if (!KEPT) {
        safe = true;
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k) {
            safe = safe && rc_safe(s[k]);
            rc[k] = rcp_exact(s[k]);
        }
    }
    return __all(safe);
}

// x[k] / s[k] with rc[k] = 1 / s[k], rounded to half where the chain is one of half ops.  Every scale is a maximum over the
// values it divides, so where all of a wave's scales lie in the range in which the reciprocal is exact (fast), one product and
// two fmas are the correctly rounded quotient.
template <bool HALF>
__device__ __forceinline__ void any_quotients(float (&x)[kAnyElts], const float (&s)[kAnyElts], const float (&rc)[kAnyElts], bool fast)
{
    if (fast) {
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k)
            x[k] = div_by_rc(x[k], s[k], rc[k]);
    } else {
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k)
            x[k] = x[k] / s[k];
    }
    if (HALF)
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k)
            x[k] = rh(x[k]);
}

template <typename REAL, bool M32, bool BITS, bool VEC>
__global__ __launch_bounds__(kThreads, 4) void rank1_requant_any_kernel(const MultiR1 args, const NewCodes out,
                                                                        const float *__restrict__ qmap_m,
                                                                        const float *__restrict__ qmap_v, int bits_m, int bits_v,
                                                                        const uint32_t *__restrict__ table_m,
                                                                        const uint32_t *__restrict__ table_v)
{
    constexpr bool HALF = sizeof(REAL) == 2;
    __shared__ typename AnyCoder<BITS>::Lds lds;
    AnyCoder<BITS> coder(lds, qmap_m, qmap_v, bits_m, bits_v, table_m, table_v);
    const int lo = find_tensor(args);
    const TensorR1 &t = args.t[lo];
    const uint32_t index = blockIdx.x - args.tile_start[lo];
    // Rows of an odd column count share bytes of the new codes: neighbouring tiles meet in atomics on the
    // words around them, and launch order, which spreads them over the XCDs, is faster (six tensors of 4095 x 4099, a step,
    // neighbours on one XCD -> here: 4 bits 965 -> 948 us, fp32 first moment 834 -> 823, float16 812 -> 791; byte codes share
    // nothing and lose 606 -> 617).
    const bool shared = !BITS && !VEC && (t.col_tail & 1) != 0;
    const uint32_t tl = shared ? index : xcd_neighbours(index, args.tile_start[lo + 1] - args.tile_start[lo]);
    const int lane16 = threadIdx.x & 15, drow = threadIdx.x >> 4;
    const Geometry q = geometry(t, tl, drow);
    const int64_t cols = (int64_t)(t.col_blocks - 1) * kGroup + t.col_tail;
    const bool odd_cols = (cols & 1) != 0;
    NfHyper h;
    h.b2 = args.b2;
    h.w2 = args.w2;
    h.w1 = args.w1;
    __syncthreads();
    coder.ready();

    const uint32_t mask_m = (1u << bits_m) - 1u, mask_v = (1u << bits_v) - 1u;
    const int lg_group = 7 + (int)t.m_lg;
    if (tl == 0) {
        const int64_t n = t.rows * cols;
        const uint32_t zero_v = coder.one(1, 0.0f);
        any_padding<BITS>(out.v[lo], n, n, zero_v, zero_v, odd_cols);
        if (!M32) {
            const int64_t group = (int64_t)1 << lg_group, n_group = (n + group - 1) / group * group;
            const float last = 0.0f / t.ms_new[(n - 1) >> lg_group];
            any_padding<BITS>(out.m[lo], n, n_group, coder.one(0, last), coder.one(0, 0.0f), odd_cols);
        }
    }
    if (q.cg >= t.col_blocks || q.row0 >= t.rows)
        return;
    const REAL *row_old = reinterpret_cast<const REAL *>(t.row_old);
    const REAL *col_old = reinterpret_cast<const REAL *>(t.col_old) + (int64_t)q.cg * kGroup;
    const float *col_new = t.col_new + (int64_t)q.cg * kGroup;
    const REAL *ms = reinterpret_cast<const REAL *>(t.ms);
    const Piece first = piece_of(cols, q.cg, q.row0, lg_group);
    REAL co[kAnyElts];
    float cn[kAnyElts], rcn[kAnyElts];
    bool cols_safe = true;
#pragma unroll
    for (int k = 0; k < kAnyElts; ++k) {
        co[k] = col_old[piece_at<VEC>(first, lane16, k)];
        cn[k] = col_new[piece_at<VEC>(first, lane16, k)];
        rcn[k] = VEC ? rcp_exact(cn[k]) : 0.0f;
        cols_safe = VEC && cols_safe && rc_safe(cn[k]);
    }
    const MixConst c = mix_const();
#pragma unroll 1
    for (int it = 0; it < q.passes; ++it) {
        const int64_t r = q.row0 + (int64_t)it * q.step;
        if (r >= t.rows)
            break;
        const Piece w = piece_of(cols, q.cg, r, lg_group);
        const REAL *gp = reinterpret_cast<const REAL *>(t.g) + w.base;
        REAL g[kAnyElts];
        float x[kAnyElts], s[kAnyElts], rc[kAnyElts];
        load_values<VEC, false>(gp, w, lane16, g);
        const uint64_t vc = load_codes<BITS, VEC>(t.vc, w, lane16);
        const uint64_t mc = M32 ? 0 : load_codes<BITS, VEC>(t.mc, w, lane16);
        const REAL ro = row_old[r];
        const float rn = t.row_new[r];
        if (!M32) {
            // runs: a piece in one group takes that group's scales twice, so that no load waits for another behind a branch
            const bool two = w.split < w.count;
            const int64_t next = w.group + (two ? 1 : 0);
            const float s0 = (float)ms[w.group], s1 = VEC ? (float)ms[next] : two ? (float)ms[w.group + 1] : 0.0f;
            const float n0 = t.ms_new[w.group], n1 = VEC ? t.ms_new[next] : two ? t.ms_new[w.group + 1] : n0;
            const float rc0 = VEC ? rcp_exact(n0) : 0.0f, rc1 = VEC ? rcp_exact(n1) : 0.0f;
#pragma unroll
            for (int k = 0; k < kAnyElts; ++k) {
                const bool here = piece_at<VEC>(w, lane16, k) < w.split;
                x[k] = any_decode<BITS>(coder.map(0), mc, k, mask_m) * (here ? s0 : s1);
                s[k] = here ? n0 : n1;
                rc[k] = here ? rc0 : rc1;
            }
            if constexpr (HALF) {
#pragma unroll
                for (int j = 0; j < kPairs; ++j) {
                    const v2h a = round2(x[2 * j], x[2 * j + 1]);
                    v2h b;
                    if (fabsf(h.w1) < 0.5f)
                        b = round2(half_lerp<true>(a.x, g[2 * j], h.w1, c), half_lerp<true>(a.y, g[2 * j + 1], h.w1, c));
                    else
                        b = round2(half_lerp<false>(a.x, g[2 * j], h.w1, c), half_lerp<false>(a.y, g[2 * j + 1], h.w1, c));
                    x[2 * j] = (float)b.x;
                    x[2 * j + 1] = (float)b.y;
                }
            } else {
#pragma unroll
                for (int k = 0; k < kAnyElts; ++k)
                    x[k] = lerp_w(x[k], g[k], h.w1);
            }
            any_quotients<HALF>(x, s, rc, any_reciprocals<VEC>(s, rc, rc_safe(n0) && rc_safe(n1)));
            coder.template store<VEC>(0, x, out.m[lo], w, lane16, odd_cols);
            // the second moment's loads stay behind the stores: 12 instead of 100 bytes of spilled registers a lane
            __builtin_amdgcn_sched_barrier(0);
        }
        const float rcr = VEC ? rcp_exact(rn) : 0.0f;
#pragma unroll
        for (int k = 0; k < kAnyElts; ++k) {
            x[k] = any_decode<BITS>(coder.map(1), vc, k, mask_v) * rank1_scale((float)co[k], (float)ro);
            const bool by_col = cn[k] < rn;
            s[k] = by_col ? cn[k] : rn;
            rc[k] = by_col ? rcn[k] : rcr;
        }
        if constexpr (HALF) {
            const RoundOnce once = rounded_once<VEC>(w, lane16, t.rows * cols, t.g);
#pragma unroll
            for (int j = 0; j < kPairs; ++j) {
                const v2h b = half_second_moment_ops(round2(x[2 * j], x[2 * j + 1]), v2h{g[2 * j], g[2 * j + 1]}, h, c, once, j);
                x[2 * j] = (float)b.x;
                x[2 * j + 1] = (float)b.y;
            }
        } else {
#pragma unroll
            for (int k = 0; k < kAnyElts; ++k)
                nonfused_second_moment(x[k], g[k], h);
        }
        any_quotients<HALF>(x, s, rc, any_reciprocals<VEC>(s, rc, cols_safe && rc_safe(rn)));
        coder.template store<VEC>(1, x, out.v[lo], w, lane16, odd_cols);
    }
}

template <typename REAL, bool M32, bool BITS, bool VEC>
static void launch_passes(const R1Launch &l, const NewCodes &out, const float *qmap_m, const float *qmap_v, int bits_m, int bits_v,
                          const uint32_t *table_m, const uint32_t *table_v, int passes, hipStream_t stream)
{
    if (passes & 1)
        hipLaunchKernelGGL((rank1_update_any_kernel<REAL, M32, BITS, VEC>), dim3(l.update_tiles), dim3(kThreads), 0, stream, l.update,
                           out, qmap_m, qmap_v, bits_m, bits_v);
    if (passes & 2)
        hipLaunchKernelGGL((rank1_requant_any_kernel<REAL, M32, BITS, VEC>), dim3(l.requant_tiles), dim3(kThreads), 0, stream,
                           l.requant, out, qmap_m, qmap_v, bits_m, bits_v, table_m, table_v);
}

template <typename REAL, bool M32, bool BITS>
static void launch(const R1Launch &l, const NewCodes &out, const float *qmap_m, const float *qmap_v, int bits_m, int bits_v,
                   const uint32_t *table_m, const uint32_t *table_v, bool runs, int passes, hipStream_t stream)
{
    if (runs)
        launch_passes<REAL, M32, BITS, true>(l, out, qmap_m, qmap_v, bits_m, bits_v, table_m, table_v, passes, stream);
    else
        launch_passes<REAL, M32, BITS, false>(l, out, qmap_m, qmap_v, bits_m, bits_v, table_m, table_v, passes, stream);
}

// Runs of four where every access of a run is whole: columns a multiple of 4, parameters, gradients and an fp32 first moment on
// boundaries of four values (code arrays lie on 4-byte boundaries in any case).
bool rank1_any_runs(const lpmm_rank1_any_tensor &t, AnyKind kind)
{
    const uintptr_t run = kind == kAnyHalf ? 8 : 16;
    return t.cols % 4 == 0 && aligned_to(t.p, run) && aligned_to(t.g, run) && (kind != kAnyFloatM || aligned_to(t.m, run));
}

void launch_rank1_any(const R1Launch &l, const NewCodes &out, const float *qmap_m, const float *qmap_v, AnyKind kind, int bits_m, int bits_v,
                      const uint32_t *table_m, const uint32_t *table_v, int passes, hipStream_t stream)
{
    switch (kind) {
    case kAnyCodes4:
        launch<float, false, false>(l, out, qmap_m, qmap_v, 4, 4, nullptr, nullptr, out.runs, passes, stream);
        break;
    case kAnyFloatM:
        launch<float, true, false>(l, out, qmap_m, qmap_v, 4, 4, nullptr, nullptr, out.runs, passes, stream);
        break;
    case kAnyBits:
        launch<float, false, true>(l, out, qmap_m, qmap_v, bits_m, bits_v, table_m, table_v, out.runs, passes, stream);
        break;
    case kAnyHalf:
        launch<h16, false, false>(l, out, qmap_m, qmap_v, 4, 4, nullptr, nullptr, out.runs, passes, stream);
        break;
    }
}

}  // namespace lpmm
