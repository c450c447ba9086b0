// Stand-alone 4-bit quantise / dequantise kernels for gfx950 in the non-fused packed layout
// of lpmm: codes of the flattened, zero-padded tensor, two per byte (low nibble = even
// index), padded to a multiple of 2048 values, plus one trailing byte
// (lpmm/functional.py:359-369, lpmm/cpp_extension/quantization_kernel.cu:430-477).
//
// A lane owns 8 consecutive values = one 32-bit word of codes; a 256-thread workgroup
// covers one 2048-value pack group.  Group maxima use DPP row reductions (128 values =
// 16 lanes) and, for larger groups, 16 floats of LDS per workgroup.  Code assignment uses
// the table / closed-form encoders of lpmm_codec.hpp when the map is one of the two
// standard ones and the count-of-midpoints search otherwise.
#include "rank1_rows.hpp"

namespace lpmm {

constexpr int kQThreads = 256;
static_assert(kQThreads == kEncEntries, "lds_fill_load / lds_fill_store: one encode-table entry per thread");
constexpr int kQElts = 8;
constexpr int kQTile = kQThreads * kQElts;  // 2048

__device__ __forceinline__ void load8(const float *__restrict__ x, int64_t base, int64_t n, bool vec,
                                      float (&v)[kQElts])
{
    if (vec && base + kQElts <= n) {
        const float4 a = load4(x + base), b = load4(x + base + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int k = 0; k < kQElts; ++k)
            v[k] = (base + k < n) ? x[base + k] : 0.0f;
    }
}

__device__ __forceinline__ void store8(float *__restrict__ out, int64_t base, int64_t n, bool vec,
                                       const float (&v)[kQElts])
{
    if (vec && base + kQElts <= n) {
        store4(out + base, make_float4(v[0], v[1], v[2], v[3]));
        store4(out + base + 4, make_float4(v[4], v[5], v[6], v[7]));
    } else {
#pragma unroll
        for (int k = 0; k < kQElts; ++k)
            if (base + k < n)
                out[base + k] = v[k];
    }
}

// codes hold at least ceil(n/2) bytes; whole words are read only where they lie inside.
__device__ __forceinline__ uint32_t load_codes8(const uint8_t *__restrict__ codes, int64_t base, int64_t n,
                                                bool vec)
{
    if (vec && base + kQElts <= n)
        return load_u32(reinterpret_cast<const uint32_t *>(codes + (base >> 1)));
    uint32_t w = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (base + 2 * k < n)
            w |= (uint32_t)codes[(base >> 1) + k] << (8 * k);
    return w;
}

// ---------------------------------------------------------------------------------------
// pack_nonlinear / unpack_nonlinear (values already normalised)
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(kQThreads) void pack4_kernel(const float *__restrict__ x,
                                                          const float *__restrict__ qmap,
                                                          int64_t n_padded, uint8_t *__restrict__ out,
                                                          bool vec)
{
    __shared__ __align__(16) uint32_t lds[kLdsBytes / 4];
    lds_fill(lds, qmap, nullptr);
    const int kind = classify_map(qmap);
    __syncthreads();
    const int64_t base = ((int64_t)blockIdx.x * kQThreads + threadIdx.x) * kQElts;
    if (base == 0)
        out[n_padded / 2] = 0;
    if (base >= n_padded)
        return;
    float v[kQElts];
    load8(x, base, n_padded, vec, v);
    const uint32_t w = encode8_plain(lds, kLdsQ0, kind, v);
    if (vec) {
        store_u32(reinterpret_cast<uint32_t *>(out + (base >> 1)), w);
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
            out[(base >> 1) + k] = (uint8_t)(w >> (8 * k));
    }
}

__global__ __launch_bounds__(kQThreads) void unpack4_kernel(const uint8_t *__restrict__ codes,
                                                            const float *__restrict__ qmap, int64_t n,
                                                            float *__restrict__ out, bool vec)
{
    __shared__ __align__(16) uint32_t lds[32];
    if (threadIdx.x < 16)
        lds[threadIdx.x] = __float_as_uint(qmap[threadIdx.x]);
    __syncthreads();
    const int64_t base = ((int64_t)blockIdx.x * kQThreads + threadIdx.x) * kQElts;
    if (base >= n)
        return;
    const Nibbles nb = split_nibbles(load_codes8(codes, base, n, vec));
    float v[kQElts];
#pragma unroll
    for (int k = 0; k < kQElts; ++k)
        v[k] = decode_nibble(lds, kLdsQ0, nb, k);
    store8(out, base, n, vec, v);
}

// ---------------------------------------------------------------------------------------
// 'group' scaling: max|x| per gp_sz values, x / max, search, pack -- one pass.
// rows_per_group = gp_sz / 128 in {1, 2, 4, 8, 16, 32}.
// ---------------------------------------------------------------------------------------
// THREADS: 256 (a tile is one 2048-value pack group) or, for gp_sz 4096, 512; a workgroup
// handles T consecutive tiles, so that the set-up of the LDS tables is paid once per T tiles.
// A workgroup whose values all lie inside the tensor (and whose operands allow vector access)
// works in the row layout of the fused step: 16 lanes own 128 consecutive values, lane l the
// values [4l, 4l+4) and [64+4l, 64+4l+4), so every 16-byte load of a row covers whole cache
// lines; the loads of all its tiles are issued before the LDS tables are set up.  Other
// workgroups (the ragged end, the padding) let every lane own 8 consecutive values and guard
// each access.
template <int THREADS, int T>
__global__ __launch_bounds__(THREADS) void quant_group_kernel(const float *__restrict__ x, int64_t n,
                                                              int rows_per_group,
                                                              const float *__restrict__ qmap,
                                                              uint8_t *__restrict__ codes,
                                                              float *__restrict__ max1, int64_t n_groups,
                                                              int64_t n_padded, bool vec)
{
    constexpr int kTileElts = THREADS * kQElts;
    __shared__ __align__(16) uint32_t lds[kLdsBytes / 4];
    __shared__ float s_row[T][THREADS / 16];
    // the workgroup's span of T tiles, in the launch order that lets an XCD stream 128 KB runs of x
    constexpr int kSpanLog2 = (T * kTileElts * sizeof(float) == 16384) ? 3 : ((T * kTileElts * sizeof(float) == 8192) ? 4 : -1);
    uint32_t span = blockIdx.x;
    if constexpr (kSpanLog2 > 0)
        span = xcd_run_order<kSpanLog2>(span, gridDim.x, run_phase<kSpanLog2>(x, T * kTileElts * sizeof(float)));
    const int64_t tile0 = (int64_t)span * T * kTileElts;
    const int lane16 = threadIdx.x & 15;
    const int wrow = threadIdx.x >> 4;
    const int64_t gp_sz = (int64_t)rows_per_group * kGroup;
    const int first = wrow & ~(rows_per_group - 1);

    if (vec && tile0 + (int64_t)T * kTileElts <= n) {  // uniform over the workgroup
        float v[T][kQElts];
        // the small loads that feed LDS first (they return first), then the tiles' loads (workgroups
        // of one thread per encode-table entry; larger ones fill the tables after their loads)
        LdsFill fill;
        if (THREADS == kEncEntries)
            fill = lds_fill_load(qmap, qmap);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const float *p = x + tile0 + (int64_t)t * kTileElts + wrow * kGroup + lane16 * 4;
            const float4 a = load4(p), b = load4(p + 64);
            v[t][0] = a.x; v[t][1] = a.y; v[t][2] = a.z; v[t][3] = a.w;
            v[t][4] = b.x; v[t][5] = b.y; v[t][6] = b.z; v[t][7] = b.w;
        }
        if (THREADS == kEncEntries)
            lds_fill_store(lds, fill);
        else
            lds_fill(lds, qmap, nullptr);
        const int kind = classify_map(qmap);
        if (tile0 == 0 && threadIdx.x == 0)
            codes[n_padded / 2] = 0;
        float amax[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            float m = 0.0f;
#pragma unroll
            for (int k = 0; k < kQElts; ++k)
                m = fmaxf(m, fabsf(v[t][k]));
            amax[t] = row16_max(m);
            if (lane16 == 0)
                s_row[t][wrow] = amax[t];
        }
        lds_barrier();
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if (rows_per_group > 1) {
                amax[t] = s_row[t][first];
                for (int r = 1; r < rows_per_group; ++r)
                    amax[t] = fmaxf(amax[t], s_row[t][first + r]);
            }
            const int64_t base = tile0 + (int64_t)t * kTileElts + wrow * kGroup;
            if ((base % gp_sz) == 0 && lane16 == 0)
                max1[base / gp_sz] = amax[t];
            const uint32_t w = encode8_scaled(lds, kLdsQ0, kind, v[t], amax[t]);
            uint16_t *cp = reinterpret_cast<uint16_t *>(codes + (base >> 1)) + lane16;
            store_u16(cp, w & 0xFFFFu);
            store_u16(cp + 16, w >> 16);
        }
        return;
    }

    lds_fill(lds, qmap, nullptr);
    const int kind = classify_map(qmap);
    if (tile0 == 0 && threadIdx.x == 0)
        codes[n_padded / 2] = 0;
    for (int t = 0; t < T; ++t) {  // uniform trip count: the barriers below are reached by all
        const int64_t base = tile0 + (int64_t)t * kTileElts + (int64_t)threadIdx.x * kQElts;
        float v[kQElts];
        load8(x, base, n, vec, v);  // zero beyond n: the reference's zero padding
        float amax = 0.0f;
#pragma unroll
        for (int k = 0; k < kQElts; ++k)
            amax = fmaxf(amax, fabsf(v[k]));
        amax = row16_max(amax);
        __syncthreads();  // the previous tile's readers are done (and, first, the tables are in)
        if (lane16 == 0)
            s_row[0][wrow] = amax;
        __syncthreads();
        if (rows_per_group > 1) {
            amax = s_row[0][first];
            for (int r = 1; r < rows_per_group; ++r)
                amax = fmaxf(amax, s_row[0][first + r]);
        }
        const int64_t grp = base / gp_sz;
        uint32_t w;
        if (grp < n_groups) {
            if ((base % gp_sz) == 0)
                max1[grp] = amax;
            w = encode8_scaled(lds, kLdsQ0, kind, v, amax);
        } else {
            // padding added by the re-grouping to 2048: plain zeros, not divided by anything
            const float z[kQElts] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            w = encode8_plain(lds, kLdsQ0, kind, z);
        }
        if (base < n_padded)  // the last workgroup may reach past the last pack group
            store_u32(reinterpret_cast<uint32_t *>(codes + (base >> 1)), w);
    }
}

__global__ __launch_bounds__(kQThreads) void dequant_group_kernel(const uint8_t *__restrict__ codes,
                                                                  const float *__restrict__ max1,
                                                                  const float *__restrict__ qmap, int64_t n,
                                                                  int64_t gp_sz, float *__restrict__ out,
                                                                  bool vec)
{
    __shared__ __align__(16) uint32_t lds[32];
    if (threadIdx.x < 16)
        lds[threadIdx.x] = __float_as_uint(qmap[threadIdx.x]);
    __syncthreads();
    const int64_t base = ((int64_t)blockIdx.x * kQThreads + threadIdx.x) * kQElts;
    if (base >= n)
        return;
    const Nibbles nb = split_nibbles(load_codes8(codes, base, n, vec));
    const float s = max1[base / gp_sz];  // gp_sz is a multiple of 128, so uniform over the lane's 8
    float v[kQElts];
#pragma unroll
    for (int k = 0; k < kQElts; ++k)
        v[k] = decode_nibble(lds, kLdsQ0, nb, k) * s;
    store8(out, base, n, vec, v);
}

// Row layout (as in the fused step): 16 lanes own one 128-value group, lane l owns values
// [4l, 4l+4) and [64+4l, 64+4l+4), so that every 16-byte store of a row covers whole cache
// lines; the values behind the last whole group go element by element.  n must be >= 128.
#ifndef LPMM_DQ_LDS_KB
#define LPMM_DQ_LDS_KB 0
#endif
// the map needs 16 words (32 allocated); more caps the workgroups resident per CU
constexpr int kDequantLdsWords = LPMM_DQ_LDS_KB > 0 ? LPMM_DQ_LDS_KB * 256 : 32;
template <int T>
__global__ __launch_bounds__(kQThreads) void dequant_group_rows_kernel(const uint8_t *__restrict__ codes,
                                                                       const float *__restrict__ max1,
                                                                       const float *__restrict__ qmap,
                                                                       int64_t full_groups, int rows_per_group,
                                                                       int64_t n, float *__restrict__ out)
{
    __shared__ __align__(16) uint32_t lds[kDequantLdsWords];
    const int lane16 = threadIdx.x & 15;
    // T passes of 16 rows each; the loads of all passes first, the map afterwards
    // the workgroup's span of T x 16 rows, in the launch order that lets an XCD stream 128 KB runs of the output
    constexpr int kSpanLog2 = (T * 2048 * sizeof(float) == 16384) ? 3 : ((T * 2048 * sizeof(float) == 8192) ? 4 : -1);
    uint32_t span = blockIdx.x;
    if constexpr (kSpanLog2 > 0)
        span = xcd_run_order<kSpanLog2>(span, gridDim.x, run_phase<kSpanLog2>(out, T * 2048 * sizeof(float)));
    const int64_t row0 = (int64_t)span * T * (kQThreads / 16) + (threadIdx.x >> 4);
    uint32_t c0[T], c1[T];
    float s[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int64_t row = row0 + t * (kQThreads / 16);
        c0[t] = c1[t] = 0;
        s[t] = 0.0f;
        if (row < full_groups) {
            const uint16_t *cp = reinterpret_cast<const uint16_t *>(codes + row * 64) + lane16;
            c0[t] = load_u16(cp);
            c1[t] = load_u16(cp + 16);
            s[t] = max1[row / rows_per_group];
        }
    }
    if (threadIdx.x < 16)
        lds[threadIdx.x] = __float_as_uint(qmap[threadIdx.x]);
    lds_barrier();
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int64_t row = row0 + t * (kQThreads / 16);
        if (row >= full_groups)
            continue;
        const Nibbles nb = split_nibbles(c0[t] | (c1[t] << 16));
        float v[kQElts];
#pragma unroll
        for (int k = 0; k < kQElts; ++k)
            v[k] = decode_nibble(lds, kLdsQ0, nb, k) * s[t];
        float *o = out + row * kGroup + lane16 * 4;
        store4(o, make_float4(v[0], v[1], v[2], v[3]));
        store4(o + 64, make_float4(v[4], v[5], v[6], v[7]));
    }
    // the values behind the last whole group: in the last workgroup instead of a launch of their own (80 million values and
    // 64: 62 + 5 -> 62 us)
    const int64_t base = full_groups * kGroup + threadIdx.x * kQElts;
    if (blockIdx.x == gridDim.x - 1 && base < n) {
        const Nibbles nb = split_nibbles(load_codes8(codes, base, n, false));
        const float scale = max1[full_groups / rows_per_group];
        float v[kQElts];
#pragma unroll
        for (int k = 0; k < kQElts; ++k)
            v[k] = decode_nibble(lds, kLdsQ0, nb, k) * scale;
        store8(out, base, n, false, v);
    }
}

// ---------------------------------------------------------------------------------------
// 'rank1' scaling of a row-major R x C tensor.
// ---------------------------------------------------------------------------------------
__global__ void fill_zero_kernel(float *__restrict__ a, int64_t na, float *__restrict__ b, int64_t nb)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < na)
        a[i] = 0.0f;
    if (i < nb)
        b[i] = 0.0f;
}

// One workgroup takes batches of 32 rows (more where a row needs fewer than 64 lanes) of a tile of up to 256 columns; a wave issues
// eight rows' loads at once, keeps its lanes' column maxima over the batches, and the waves' column maxima meet in LDS: one
// atomic per column and tile (a maximum is exact and order-free).  Atomics on one address are served one after the other, about
// 18 ns each, so a column may have one tile per 40000 values of the tensor at most: half the time that reading them takes.  One
// batch a tile where that allows it: the many small workgroups then keep the memory system busy the way a plain streaming read does.
// Measured, against one batch a tile of 256 columns and (40000 x 1601) a kernel of 1024 columns with one load a value:
// 524288 x 128 311.6 -> 56.0 us, 1000000 x 20 361.4 -> 25.2, 40000 x 1601 173.7 -> 58.3; 50257 x 1600 54.5 -> 55.0, 16384 x 4096
// 46.6 -> 45.2.
constexpr int kStatBatch = 8;                                    // loads of a lane in flight
constexpr int kStatTileRows = (kQThreads / kWave) * kStatBatch;  // rows of a batch with one row a load

// More rows are refused, as they always were: callers may count on the status.
constexpr int64_t kStatMaxRows = 65535LL * 64;

struct StatShape {
    uint32_t tiles_x;  // column tiles
    uint32_t lg_lanes; // lanes that share a row: a tile is 4 << lg_lanes columns wide
    uint32_t batches;
};

template <bool VEC>
__global__ __launch_bounds__(kQThreads) void rank1_stats_tile_kernel(const float *__restrict__ x, int64_t R, int64_t C,
                                                                     const StatShape sh, float *__restrict__ rowmax,
                                                                     float *__restrict__ colmax)
{
    __shared__ uint32_t s_col[4 * kWave];
    const uint32_t ty = blockIdx.x / sh.tiles_x, tx = blockIdx.x - ty * sh.tiles_x;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    const int lanes = 1 << sh.lg_lanes, sub = kWave >> sh.lg_lanes;
    const int sl = lane & (lanes - 1), sr = lane >> sh.lg_lanes;
    const int64_t tile_c0 = (int64_t)tx * (4 * lanes);
    // VEC: four neighbouring columns a lane; otherwise four that lie `lanes` apart
    const int64_t c0 = tile_c0 + (VEC ? sl * 4 : sl), c_step = VEC ? 1 : lanes;
    const bool cols_in = c0 + 3 * c_step < C;
    s_col[threadIdx.x] = 0u;
    float cm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t it = 0; it < sh.batches; ++it) {
        const int64_t first = ((int64_t)ty * sh.batches + it) * (kStatTileRows * sub) + (int64_t)wave * (kStatBatch * sub);
        if (first >= R)
            break;
        float a[kStatBatch][4];
        if (cols_in && first + kStatBatch * sub <= R) {
            const float *base = x + (first + sr) * C + c0;
            const int64_t step = (int64_t)sub * C;
#pragma unroll
            for (int u = 0; u < kStatBatch; ++u) {
                if (VEC) {
                    const float4 t = load4(base + u * step);
                    a[u][0] = t.x; a[u][1] = t.y; a[u][2] = t.z; a[u][3] = t.w;
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        a[u][k] = __builtin_nontemporal_load(base + u * step + k * c_step);
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < kStatBatch; ++u) {
                const int64_t r = first + u * sub + sr;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    a[u][k] = (r < R && c0 + k * c_step < C) ? x[r * C + c0 + k * c_step] : 0.0f;
            }
        }
        float rm[kStatBatch];
#pragma unroll
        for (int u = 0; u < kStatBatch; ++u) {
            const float a0 = fabsf(a[u][0]), a1 = fabsf(a[u][1]), a2 = fabsf(a[u][2]), a3 = fabsf(a[u][3]);
            rm[u] = fmaxf(fmaxf(a0, a1), fmaxf(a2, a3));
            cm[0] = fmaxf(cm[0], a0);
            cm[1] = fmaxf(cm[1], a1);
            cm[2] = fmaxf(cm[2], a2);
            cm[3] = fmaxf(cm[3], a3);
        }
        if (lanes == kWave) {
            const float m = wave_max8(rm, lane);  // lane 8u: maximum of row first + u over the tile's columns
            const int64_t r = first + (lane >> 3);
            if ((lane & 7) == 0 && r < R) {
                if (sh.tiles_x == 1)
                    rowmax[r] = m;
                else
                    atomic_max_nonneg(rowmax + r, m);
            }
        } else {
            // a tile this narrow is the whole row; no maximum is below zero, so that a row of NaNs alone has zero, as it has
            // where lanes without columns take part
#pragma unroll
            for (int u = 0; u < kStatBatch; ++u)
                rm[u] = fmaxf(rm[u], 0.0f);
            for (int o = lanes >> 1; o > 0; o >>= 1) {
#pragma unroll
                for (int u = 0; u < kStatBatch; ++u)
                    rm[u] = fmaxf(rm[u], __shfl_xor(rm[u], o, kWave));
            }
#pragma unroll
            for (int u = 0; u < kStatBatch; ++u) {
                const int64_t r = first + u * sub + sr;
                if (sl == (u & (lanes - 1)) && r < R)
                    rowmax[r] = rm[u];
            }
        }
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < 4; ++k)
        atomicMax(s_col + (VEC ? sl * 4 + k : sl + k * lanes), __float_as_uint(cm[k]));
    lds_barrier();
    if (threadIdx.x < 4u * lanes && tile_c0 + threadIdx.x < C)
        atomic_max_nonneg(colmax + tile_c0 + threadIdx.x, __uint_as_float(s_col[threadIdx.x]));
}

// Normalise by min(rowmax[r], colmax[c]), search, pack.  Flattened indexing: a lane's 8
// values may straddle rows (any C).
__global__ __launch_bounds__(kQThreads) void quant_rank1_kernel(const float *__restrict__ x, int64_t n,
                                                                int64_t C, const float *__restrict__ rowmax,
                                                                const float *__restrict__ colmax,
                                                                const float *__restrict__ qmap,
                                                                uint8_t *__restrict__ codes, int64_t n_padded,
                                                                bool vec)
{
    __shared__ __align__(16) uint32_t lds[kLdsBytes / 4];
    lds_fill(lds, qmap, nullptr);
    const int kind = classify_map(qmap);
    __syncthreads();
    const int64_t base = ((int64_t)blockIdx.x * kQThreads + threadIdx.x) * kQElts;
    if (base == 0)
        codes[n_padded / 2] = 0;
    float v[kQElts], xs[kQElts];
    load8(x, base, n, vec, v);
    int64_t r = base / C;
    int64_t c = base - r * C;
    float rm = (base < n) ? rowmax[r] : 0.0f;
#pragma unroll
    for (int k = 0; k < kQElts; ++k) {
        xs[k] = 0.0f;  // padding added by the re-grouping to 2048
        if (base + k < n) {
            const float cmx = colmax[c];
            const float st = (cmx < rm) ? cmx : rm;
            xs[k] = v[k] / st;
            if (++c == C) {
                c = 0;
                ++r;
                rm = (base + k + 1 < n) ? rowmax[r] : 0.0f;
            }
        }
    }
    store_u32(reinterpret_cast<uint32_t *>(codes + (base >> 1)), encode8_plain(lds, kLdsQ0, kind, xs));
}

// Codes of v[k] / min(cmx[k], rm) for a lane's 8 values of one row.  The column maxima stay the
// same for every row a lane handles, so their correctly rounded reciprocals are formed once
// (col_rcp); with the row's reciprocal that turns every division into one multiply and two fmas
// that give the correctly rounded quotient.  Scales outside the range in which the reciprocal is
// exact, maps other than the two standard ones and values far beyond their statistics (rc_covers)
// take the plain division.
struct ColRcp {
    float rc[kQElts];
    bool safe;
};

__device__ __forceinline__ ColRcp col_rcp(const float (&cmx)[kQElts])
{
    ColRcp c;
    c.safe = true;
#pragma unroll
    for (int k = 0; k < kQElts; ++k) {
        c.rc[k] = rcp_exact(cmx[k]);
        c.safe = c.safe && rc_safe(cmx[k]);
    }
    return c;
}

__device__ __forceinline__ uint32_t encode8_rank1(const uint32_t *lds, int kind, const float (&v)[kQElts],
                                                  const float (&cmx)[kQElts], const ColRcp &cr, float rm)
{
    float xs[kQElts];
    if (kind != kMapGeneric && __all(cr.safe & rc_safe(rm) & rc_covers(v))) {
        const float rr = rcp_exact(rm);
#pragma unroll
        for (int k = 0; k < kQElts; ++k) {
            const bool by_col = cmx[k] < rm;
            xs[k] = div_by_rc(v[k], by_col ? cmx[k] : rm, by_col ? cr.rc[k] : rr);
        }
        // the closed form of the second-moment code needs 0 <= x <= 1; other values are legal here
        return kind == kMapStdM ? encode8_std_m(lds, xs) : encode8_plain(lds, kLdsQ0, kind, xs);
    }
#pragma unroll
    for (int k = 0; k < kQElts; ++k)
        xs[k] = v[k] / ((cmx[k] < rm) ? cmx[k] : rm);
    return encode8_plain(lds, kLdsQ0, kind, xs);
}

template <bool ONE>
__global__ __launch_bounds__(kQThreads) void quant_rank1_rows_kernel(const float *__restrict__ x, int64_t R, int64_t C,
                                                                     const RowShape sh, const float *__restrict__ rowmax,
                                                                     const float *__restrict__ colmax,
                                                                     const float *__restrict__ qmap,
                                                                     uint8_t *__restrict__ codes, int64_t n_padded)
{
    constexpr int T = kR1RowsPerWg;
    __shared__ __align__(16) uint32_t lds[kLdsBytes / 4];
    const int64_t n = R * C;
    const RowLane q = row_lane<ONE>(sh, C);
    // the small loads that feed LDS first (they return first), then the rows' loads
    const LdsFill fill = lds_fill_load(qmap, qmap);
    float4 a[T], b[T], ca, cb;
    float rm[T];
    ca = *reinterpret_cast<const float4 *>(colmax + q.c);
    cb = *reinterpret_cast<const float4 *>(colmax + q.c2);
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int64_t r_in = row_of<ONE>(q, sh, t), r = r_in < R ? r_in : R - 1;
        a[t] = load4(x + r * C + q.c);
        b[t] = load4(x + r * C + q.c2);
        rm[t] = rowmax[r];
    }
    lds_fill_store(lds, fill);
    const int kind = classify_map(qmap);
    lds_barrier();
    if (blockIdx.x == 0 && blockIdx.y == 0) {
        const float z[kQElts] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        const uint32_t wz = encode8_plain(lds, kLdsQ0, kind, z);
        // n is a multiple of 4 here: its first run of padding is half a word
        if (threadIdx.x == 0 && n < n_padded && (n & 4) != 0)
            *reinterpret_cast<uint16_t *>(codes + (n >> 1)) = (uint16_t)wz;
        for (int64_t i = (n + 7) / 8 * 8 + (int64_t)threadIdx.x * kQElts; i < n_padded; i += kR1Cols)
            *reinterpret_cast<uint32_t *>(codes + (i >> 1)) = wz;
        if (threadIdx.x == 0)
            codes[n_padded / 2] = 0;
    }
    if (!q.live)
        return;
    const float cmx[kQElts] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
    const ColRcp cr = col_rcp(cmx);
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int64_t r = row_of<ONE>(q, sh, t);
        if (r >= R)
            break;
        const float v[kQElts] = {a[t].x, a[t].y, a[t].z, a[t].w, b[t].x, b[t].y, b[t].z, b[t].w};
        const uint32_t w = encode8_rank1(lds, kind, v, cmx, cr, rm[t]);
        uint16_t *cp = reinterpret_cast<uint16_t *>(codes + ((r * C + q.c) >> 1));
        store_u16(cp, w & 0xFFFFu);
        if (q.second)
            store_u16(cp + kRowHalf / 4, w >> 16);
    }
}

__global__ __launch_bounds__(kQThreads) void dequant_rank1_kernel(const uint8_t *__restrict__ codes,
                                                                  const float *__restrict__ rowmax,
                                                                  const float *__restrict__ colmax,
                                                                  const float *__restrict__ qmap, int64_t n,
                                                                  int64_t C, float *__restrict__ out, bool vec)
{
    __shared__ __align__(16) uint32_t lds[32];
    if (threadIdx.x < 16)
        lds[threadIdx.x] = __float_as_uint(qmap[threadIdx.x]);
    __syncthreads();
    const int64_t base = ((int64_t)blockIdx.x * kQThreads + threadIdx.x) * kQElts;
    if (base >= n)
        return;
    const Nibbles nb = split_nibbles(load_codes8(codes, base, n, vec));
    int64_t r = base / C;
    int64_t c = base - r * C;
    float rm = rowmax[r];
    float v[kQElts];
#pragma unroll
    for (int k = 0; k < kQElts; ++k) {
        v[k] = 0.0f;
        if (base + k < n) {
            const float cmx = colmax[c];
            const float st = (cmx < rm) ? cmx : rm;
            v[k] = decode_nibble(lds, kLdsQ0, nb, k) * st;
            if (++c == C) {
                c = 0;
                ++r;
                rm = (base + k + 1 < n) ? rowmax[r] : 0.0f;
            }
        }
    }
    store8(out, base, n, vec, v);
}

// columns a multiple of 128: every lane has its second run, one without work too (that of column 0).  Not to choose its place as
// row_lane does: 8192 x 8192 57.2 -> 55.2 us, 32768 x 2048 57.9 -> 55.3
template <bool ONE>
__global__ __launch_bounds__(kQThreads) void dequant_rank1_rows_kernel(const uint8_t *__restrict__ codes,
                                                                       const float *__restrict__ rowmax,
                                                                       const float *__restrict__ colmax,
                                                                       const float *__restrict__ qmap, int64_t R,
                                                                       int64_t C, const RowShape sh, float *__restrict__ out)
{
    constexpr int T = kR1RowsPerWg;
    __shared__ __align__(16) uint32_t lds[32];
    const RowLane q = row_lane<ONE>(sh, C);
    uint32_t w0[T], w1[T];
    float rm[T];
    float4 ca, cb;
    ca = *reinterpret_cast<const float4 *>(colmax + q.c);
    cb = *reinterpret_cast<const float4 *>(colmax + q.c + kRowHalf);
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int64_t r_in = row_of<ONE>(q, sh, t), r = r_in < R ? r_in : R - 1;
        w0[t] = load_u16(reinterpret_cast<const uint16_t *>(codes + ((r * C + q.c) >> 1)));
        w1[t] = load_u16(reinterpret_cast<const uint16_t *>(codes + ((r * C + q.c) >> 1)) + kRowHalf / 4);
        rm[t] = rowmax[r];
    }
    if (threadIdx.x < 16)
        lds[threadIdx.x] = __float_as_uint(qmap[threadIdx.x]);
    lds_barrier();
    if (!q.live)
        return;
    const float cmx[kQElts] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int64_t r = row_of<ONE>(q, sh, t);
        if (r >= R)
            break;
        const Nibbles nb = split_nibbles(w0[t] | (w1[t] << 16));
        float v[kQElts];
#pragma unroll
        for (int k = 0; k < kQElts; ++k)
            v[k] = decode_nibble(lds, kLdsQ0, nb, k) * ((cmx[k] < rm[t]) ? cmx[k] : rm[t]);
        float *o = out + r * C + q.c;
        store4(o, make_float4(v[0], v[1], v[2], v[3]));
        store4(o + kRowHalf, make_float4(v[4], v[5], v[6], v[7]));
    }
}

template <bool RUNS>
__global__ __launch_bounds__(kQThreads) void quant_rank1_flat_kernel(const float *__restrict__ x, int64_t n, const FlatCols f,
                                                                     const float *__restrict__ rowmax,
                                                                     const float *__restrict__ colmax,
                                                                     const float *__restrict__ qmap,
                                                                     uint8_t *__restrict__ codes, int64_t n_padded)
{
    __shared__ __align__(16) uint32_t lds[kLdsBytes / 4];
    const int64_t b0 = (int64_t)flat_tile(x) * kFlatTile;
    const bool whole = b0 + kFlatTile <= n;
    const LdsFill fill = lds_fill_load(qmap, qmap);
    float4 a[kFlatT];
    FlatStats<RUNS> st[kFlatT];
    flat_load<RUNS>(x, b0, n, whole, a);
    flat_stats_of_tile<RUNS>(rowmax, colmax, b0, n, whole, f, st);
    lds_fill_store(lds, fill);
    const int kind = classify_map(qmap);
    lds_barrier();
    if (b0 == 0 && threadIdx.x == 0)
        codes[n_padded / 2] = 0;
#pragma unroll
    for (int t = 0; t < kFlatT; t += 2) {
        const int64_t i0 = b0 + t * kFlatPass + threadIdx.x * 4, i1 = i0 + kFlatPass;
        const float v[kQElts] = {a[t].x, a[t].y, a[t].z, a[t].w, a[t + 1].x, a[t + 1].y, a[t + 1].z, a[t + 1].w};
        float s[kQElts], xs[kQElts];
        flat_scales<RUNS>(st[t], s);
        flat_scales<RUNS>(st[t + 1], s + 4);
        bool safe = kind != kMapGeneric;
#pragma unroll
        for (int k = 0; k < kQElts; ++k)
            safe = safe && rc_safe(s[k]);
        const bool fast = __all(safe) && __all(rc_covers(v));
        if (fast) {
#pragma unroll
            for (int k = 0; k < kQElts; ++k)
                xs[k] = div_by_rc(v[k], s[k], rcp_exact(s[k]));
        } else {
            // the values that pad the tensor are plain zeros
#pragma unroll
            for (int k = 0; k < kQElts; ++k) {
                const int64_t i = (k < 4 ? i0 : i1) + (k & 3);
                xs[k] = i < n ? v[k] / s[k] : 0.0f;
            }
        }
        const uint32_t w = fast && kind == kMapStdM ? encode8_std_m(lds, xs) : encode8_plain(lds, kLdsQ0, kind, xs);
        if (whole || i0 < n_padded)
            store_u16(reinterpret_cast<uint16_t *>(codes + (i0 >> 1)), w & 0xFFFFu);
        if (whole || i1 < n_padded)
            store_u16(reinterpret_cast<uint16_t *>(codes + (i1 >> 1)), w >> 16);
    }
}

template <bool RUNS>
__global__ __launch_bounds__(kQThreads) void dequant_rank1_flat_kernel(const uint8_t *__restrict__ codes, int64_t n,
                                                                       const FlatCols f, const float *__restrict__ rowmax,
                                                                       const float *__restrict__ colmax,
                                                                       const float *__restrict__ qmap, float *__restrict__ out)
{
    __shared__ __align__(16) uint32_t lds[32];
    const int64_t b0 = (int64_t)flat_tile(out) * kFlatTile;
    const bool whole = b0 + kFlatTile <= n;
    uint32_t w[kFlatT];
    FlatStats<RUNS> st[kFlatT];
#pragma unroll
    for (int t = 0; t < kFlatT; ++t) {
        const int64_t idx = b0 + t * kFlatPass + threadIdx.x * 4;
        w[t] = 0;
        if (whole || idx + 4 <= n)
            w[t] = load_u16(reinterpret_cast<const uint16_t *>(codes + (idx >> 1)));
        else if (!RUNS && idx < n)
            w[t] = codes[idx >> 1] | (idx + 2 < n ? (uint32_t)codes[(idx >> 1) + 1] << 8 : 0u);
    }
    flat_stats_of_tile<RUNS>(rowmax, colmax, b0, n, whole, f, st);
    if (threadIdx.x < 16)
        lds[threadIdx.x] = __float_as_uint(qmap[threadIdx.x]);
    lds_barrier();
#pragma unroll
    for (int t = 0; t < kFlatT; t += 2) {
        const Nibbles nb = split_nibbles(w[t] | (w[t + 1] << 16));
        float s[kQElts], v[kQElts];
        flat_scales<RUNS>(st[t], s);
        flat_scales<RUNS>(st[t + 1], s + 4);
#pragma unroll
        for (int k = 0; k < kQElts; ++k)
            v[k] = decode_nibble(lds, kLdsQ0, nb, k) * s[k];
        flat_store<RUNS>(out, b0 + t * kFlatPass + threadIdx.x * 4, n, whole, v);
        flat_store<RUNS>(out, b0 + (t + 1) * kFlatPass + threadIdx.x * 4, n, whole, v + 4);
    }
}

inline bool tiles_ok(int64_t n, int64_t tile, uint32_t *tiles)
{
    const int64_t t = (n + tile - 1) / tile;
    if (t > 0x7fffffffLL)
        return false;
    *tiles = (uint32_t)t;
    return true;
}

}  // namespace lpmm

using namespace lpmm;

extern "C" int lpmm_pack_nonlinear_4bit(const float *x, const float *qmap, int64_t n_padded,
                                        uint8_t *out, void *stream)
{
    if (n_padded < 0 || (n_padded % 8) != 0)
        return LPMM_ERR_SIZE;
    LPMM_REQUIRE_PTR(out);
    LPMM_REQUIRE_PTR(qmap);
    LPMM_REQUIRE_ALIGN(qmap, 4);
    if (n_padded > 0) {
        LPMM_REQUIRE_PTR(x);
        LPMM_REQUIRE_ALIGN(x, 4);
    }
    uint32_t tiles;
    if (!tiles_ok(n_padded > 0 ? n_padded : 1, kQTile, &tiles))
        return LPMM_ERR_SIZE;
    const bool vec = aligned_to(x, 16) && aligned_to(out, 4);
    hipLaunchKernelGGL(pack4_kernel, dim3(tiles), dim3(kQThreads), 0, (hipStream_t)stream, x, qmap,
                       n_padded, out, vec);
    return launch_status();
}

extern "C" int lpmm_unpack_nonlinear_4bit(const uint8_t *codes, const float *qmap, int64_t n,
                                          float *out, void *stream)
{
    if (n < 0)
        return LPMM_ERR_SIZE;
    if (n == 0)
        return LPMM_OK;
    LPMM_REQUIRE_PTR(codes);
    LPMM_REQUIRE_PTR(qmap);
    LPMM_REQUIRE_PTR(out);
    LPMM_REQUIRE_ALIGN(qmap, 4);
    LPMM_REQUIRE_ALIGN(out, 4);
    uint32_t tiles;
    if (!tiles_ok(n, kQTile, &tiles))
        return LPMM_ERR_SIZE;
    const bool vec = aligned_to(out, 16) && aligned_to(codes, 4);
    hipLaunchKernelGGL(unpack4_kernel, dim3(tiles), dim3(kQThreads), 0, (hipStream_t)stream, codes, qmap,
                       n, out, vec);
    return launch_status();
}

extern "C" int lpmm_quant_group(const float *x, int64_t n, int64_t gp_sz, const float *qmap,
                                uint8_t *codes, float *max1, void *stream)
{
    if (n <= 0)
        return LPMM_ERR_SIZE;
    if (gp_sz < kGroup || gp_sz > 2 * kQTile || (gp_sz & (gp_sz - 1)) != 0)
        return LPMM_ERR_SIZE;
    LPMM_REQUIRE_PTR(x);
    LPMM_REQUIRE_PTR(qmap);
    LPMM_REQUIRE_PTR(codes);
    LPMM_REQUIRE_PTR(max1);
    LPMM_REQUIRE_ALIGN(x, 4);
    LPMM_REQUIRE_ALIGN(qmap, 4);
    LPMM_REQUIRE_ALIGN(max1, 4);
    LPMM_REQUIRE_ALIGN(codes, 4);
    const int64_t n_groups = (n + gp_sz - 1) / gp_sz;
    uint32_t tiles;
    if (!tiles_ok(n_groups * gp_sz, kQTile, &tiles))
        return LPMM_ERR_SIZE;
    const int64_t n_padded = (int64_t)tiles * kQTile;
#ifndef LPMM_QG_T
#define LPMM_QG_T 2
#endif
    constexpr int kT = LPMM_QG_T;  // tiles per workgroup
    if (gp_sz > kQTile)
        hipLaunchKernelGGL((quant_group_kernel<2 * kQThreads, 1>), dim3((tiles + 1) / 2), dim3(2 * kQThreads), 0,
                           (hipStream_t)stream, x, n, (int)(gp_sz / kGroup), qmap, codes, max1, n_groups, n_padded,
                           aligned_to(x, 16));
    else
        hipLaunchKernelGGL((quant_group_kernel<kQThreads, kT>), dim3((tiles + kT - 1) / kT), dim3(kQThreads), 0,
                           (hipStream_t)stream, x, n, (int)(gp_sz / kGroup), qmap, codes, max1, n_groups, n_padded,
                           aligned_to(x, 16));
    return launch_status();
}

extern "C" int lpmm_dequant_group(const uint8_t *codes, const float *max1, const float *qmap, int64_t n,
                                  int64_t gp_sz, float *out, void *stream)
{
    if (n <= 0 || gp_sz < kGroup || (gp_sz % kGroup) != 0)
        return LPMM_ERR_SIZE;
    LPMM_REQUIRE_PTR(codes);
    LPMM_REQUIRE_PTR(max1);
    LPMM_REQUIRE_PTR(qmap);
    LPMM_REQUIRE_PTR(out);
    LPMM_REQUIRE_ALIGN(max1, 4);
    LPMM_REQUIRE_ALIGN(qmap, 4);
    LPMM_REQUIRE_ALIGN(out, 4);
    uint32_t tiles;
    if (!tiles_ok(n, kQTile, &tiles))
        return LPMM_ERR_SIZE;
    const bool vec = aligned_to(out, 16) && aligned_to(codes, 4);
    const int64_t full_groups = n / kGroup;
    if (vec && full_groups > 0 && full_groups <= 0x7fffffffLL * 16) {
#ifndef LPMM_DQ_T
#define LPMM_DQ_T 2
#endif
        constexpr int kT = LPMM_DQ_T;  // passes of 16 rows per workgroup
        hipLaunchKernelGGL(dequant_group_rows_kernel<kT>, dim3((uint32_t)((full_groups + 16 * kT - 1) / (16 * kT))),
                           dim3(kQThreads), 0, (hipStream_t)stream, codes, max1, qmap, full_groups,
                           (int)(gp_sz / kGroup), n, out);
        return launch_status();
    }
    hipLaunchKernelGGL(dequant_group_kernel, dim3(tiles), dim3(kQThreads), 0, (hipStream_t)stream, codes,
                       max1, qmap, n, gp_sz, out, vec);
    return launch_status();
}

extern "C" int lpmm_rank1_stats(const float *x, int64_t rows, int64_t cols, float *rowmax, float *colmax,
                                void *stream)
{
    if (rows <= 0 || cols <= 0)
        return LPMM_ERR_SIZE;
    LPMM_REQUIRE_PTR(x);
    LPMM_REQUIRE_PTR(rowmax);
    LPMM_REQUIRE_PTR(colmax);
    LPMM_REQUIRE_ALIGN(x, 4);
    LPMM_REQUIRE_ALIGN(rowmax, 4);
    LPMM_REQUIRE_ALIGN(colmax, 4);
    StatShape sh;
    sh.lg_lanes = 6;
    while (sh.lg_lanes > 0 && (4LL << (sh.lg_lanes - 1)) >= cols)
        --sh.lg_lanes;
    const int64_t tx = (cols - 1) / (4LL << sh.lg_lanes) + 1;
    if (tx > 0x7fffffffLL || rows > kStatMaxRows)
        return LPMM_ERR_SIZE;
    const int64_t batch_rows = (int64_t)kStatTileRows * (kWave >> sh.lg_lanes), row_batches = (rows + batch_rows - 1) / batch_rows;
    // tiles on a column: see rank1_stats_tile_kernel; and no more than a grid holds
    int64_t most = rows * cols / 40000 > 256 ? rows * cols / 40000 : 256;
    most = most < 0x7fffffffLL / tx ? most : 0x7fffffffLL / tx;
    sh.tiles_x = (uint32_t)tx;
    sh.batches = (uint32_t)((row_batches + most - 1) / most);
    const int64_t tiles = tx * ((row_batches + sh.batches - 1) / sh.batches);
    const int64_t mx = rows > cols ? rows : cols;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((uint32_t)((mx + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, rowmax, rows, colmax, cols);
    if (aligned_to(x, 16) && (cols % 4) == 0)
        hipLaunchKernelGGL(rank1_stats_tile_kernel<true>, dim3((uint32_t)tiles), dim3(kQThreads), 0, (hipStream_t)stream, x, rows,
                           cols, sh, rowmax, colmax);
    else
        hipLaunchKernelGGL(rank1_stats_tile_kernel<false>, dim3((uint32_t)tiles), dim3(kQThreads), 0, (hipStream_t)stream, x, rows,
                           cols, sh, rowmax, colmax);
    return launch_status();
}

extern "C" int lpmm_quant_rank1(const float *x, int64_t rows, int64_t cols, const float *rowmax,
                                const float *colmax, const float *qmap, uint8_t *codes, void *stream)
{
    if (rows <= 0 || cols <= 0)
        return LPMM_ERR_SIZE;
    LPMM_REQUIRE_PTR(x);
    LPMM_REQUIRE_PTR(rowmax);
    LPMM_REQUIRE_PTR(colmax);
    LPMM_REQUIRE_PTR(qmap);
    LPMM_REQUIRE_PTR(codes);
    LPMM_REQUIRE_ALIGN(x, 4);
    LPMM_REQUIRE_ALIGN(rowmax, 4);
    LPMM_REQUIRE_ALIGN(colmax, 4);
    LPMM_REQUIRE_ALIGN(qmap, 4);
    LPMM_REQUIRE_ALIGN(codes, 4);
    const int64_t n = rows * cols;
    uint32_t tiles;
    if (!tiles_ok(n, kQTile, &tiles))
        return LPMM_ERR_SIZE;
    const int64_t n_padded = (int64_t)tiles * kQTile;
    RowShape sh;
    dim3 rows_grid;
    if (rank1_rows(x, colmax, codes, rows, cols, true, sh, rows_grid)) {
        const auto kernel = sh.groups == 1 ? quant_rank1_rows_kernel<true> : quant_rank1_rows_kernel<false>;
        hipLaunchKernelGGL(kernel, rows_grid, dim3(kQThreads), 0, (hipStream_t)stream, x, rows, cols, sh, rowmax,
                           colmax, qmap, codes, n_padded);
    } else if (rank1_flat_ok(x, colmax, codes, cols)) {
        const dim3 grid((uint32_t)((n_padded + kFlatTile - 1) / kFlatTile));
        if (cols % 4 == 0)
            hipLaunchKernelGGL(quant_rank1_flat_kernel<true>, grid, dim3(kQThreads), 0, (hipStream_t)stream, x, n, flat_cols(cols),
                               rowmax, colmax, qmap, codes, n_padded);
        else
            hipLaunchKernelGGL(quant_rank1_flat_kernel<false>, grid, dim3(kQThreads), 0, (hipStream_t)stream, x, n, flat_cols(cols),
                               rowmax, colmax, qmap, codes, n_padded);
    } else {
        hipLaunchKernelGGL(quant_rank1_kernel, dim3(tiles), dim3(kQThreads), 0, (hipStream_t)stream, x, n, cols,
                           rowmax, colmax, qmap, codes, n_padded, aligned_to(x, 16));
    }
    return launch_status();
}

extern "C" int lpmm_dequant_rank1(const uint8_t *codes, const float *rowmax, const float *colmax,
                                  const float *qmap, int64_t rows, int64_t cols, float *out, void *stream)
{
    if (rows <= 0 || cols <= 0)
        return LPMM_ERR_SIZE;
    LPMM_REQUIRE_PTR(codes);
    LPMM_REQUIRE_PTR(rowmax);
    LPMM_REQUIRE_PTR(colmax);
    LPMM_REQUIRE_PTR(qmap);
    LPMM_REQUIRE_PTR(out);
    LPMM_REQUIRE_ALIGN(rowmax, 4);
    LPMM_REQUIRE_ALIGN(colmax, 4);
    LPMM_REQUIRE_ALIGN(qmap, 4);
    LPMM_REQUIRE_ALIGN(out, 4);
    const int64_t n = rows * cols;
    uint32_t tiles;
    if (!tiles_ok(n, kQTile, &tiles))
        return LPMM_ERR_SIZE;
    RowShape sh;
    dim3 rows_grid;
    if (rank1_rows(out, colmax, codes, rows, cols, false, sh, rows_grid)) {
        const auto kernel = sh.groups == 1 ? dequant_rank1_rows_kernel<true> : dequant_rank1_rows_kernel<false>;
        hipLaunchKernelGGL(kernel, rows_grid, dim3(kQThreads), 0, (hipStream_t)stream, codes, rowmax, colmax, qmap,
                           rows, cols, sh, out);
    } else if (rank1_flat_ok(out, colmax, codes, cols)) {
        const dim3 grid((uint32_t)((n + kFlatTile - 1) / kFlatTile));
        if (cols % 4 == 0)
            hipLaunchKernelGGL(dequant_rank1_flat_kernel<true>, grid, dim3(kQThreads), 0, (hipStream_t)stream, codes, n,
                               flat_cols(cols), rowmax, colmax, qmap, out);
        else
            hipLaunchKernelGGL(dequant_rank1_flat_kernel<false>, grid, dim3(kQThreads), 0, (hipStream_t)stream, codes, n,
                               flat_cols(cols), rowmax, colmax, qmap, out);
    } else {
        const bool vec = aligned_to(out, 16) && aligned_to(codes, 4);
        hipLaunchKernelGGL(dequant_rank1_kernel, dim3(tiles), dim3(kQThreads), 0, (hipStream_t)stream, codes,
                           rowmax, colmax, qmap, n, cols, out, vec);
    }
    return launch_status();
}
