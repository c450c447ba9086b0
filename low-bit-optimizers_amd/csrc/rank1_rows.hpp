// Work split of the 'rank1' quantisers and dequantisers (quantize.hip: 4 bits, quantize_bits.hip: one code per byte) over a
// row-major R x C matrix whose value (r, c) has the scale min(rowmax[r], colmax[c]).  Two splits, both in runs of four values
// (16 bytes) that are neighbours in neighbouring lanes, so that a wave's access covers whole cache lines:
//
//   rows   a lane keeps eight columns (two runs, 64 columns apart) over kR1RowsPerWg rows, so that the columns' statistics and
//          their reciprocals are formed once; narrow matrices have several rows side by side;
//   flat   a workgroup takes 16 KB of consecutive values, in the tile order of xcd_run_order; a lane works out row and column of
//          each of its runs and reads their statistics from the cache.  Every access is whole whatever C is.
//
// Measured, 4 bits (us, quantise / dequantise; "before": lanes of 8 neighbouring values for columns that are a multiple of 8,
// one division of the index and plain divisions for other columns, 16 lanes to 128 columns for multiples of 128):
//                     rows          flat          before
//   50257 x 1600      62.8 / 80.4   78.5 / 72.7   73.8 / 99.2
//   16384 x 4096      47.9 / 55.1   70.4 / 68.4   47.8 / 57.0
//   524288 x 128      48.2 / 54.5   63.6 / 56.7   157.5 / 152.3
//   20000 x 1000      18.8 / 22.0   23.3 / 20.2   24.4 / 29.0
//   40000 x 500       18.4 / 24.2   22.8 / 19.3   49.7 / 46.5
//   60000 x 300       24.2 / 28.2   21.7 / 17.4   45.1 / 42.7
//   200000 x 100      22.8 / 29.6   24.0 / 19.6
//   1000000 x 20      25.3 / 41.9   21.3 / 19.0   33.7 / 30.7
//   40000 x 1601                    87.7 / 91.2   136.4 / 145.1
// 8 bits, the same order: 72.7 / 73.0 against 210.1 / 177.3 on the first shape, 85.7 / 90.0 against 148.6 / 133.0 on the last.
// A quantiser divides, so the reciprocals kept over the rows decide; a dequantiser only writes, and rows of columns that are no
// multiple of 128 cut its lines.  No lane branches around a load: with a branch for each run and row the quantiser takes 72.0
// on the first shape and 57.2 on the second.  2 or 8 rows a lane: 70.0 and 77.5 against 72.1 there, 58.7 and 58.0 against
// 57.1; flat tiles of 8 or 32 KB: 91.8 / 73.4 and 81.7 / 71.9 on the first shape.
#pragma once
#include "lpmm_codec.hpp"

namespace lpmm {

constexpr int kRank1Threads = 256;

// ---- rows -------------------------------------------------------------------------------
constexpr int kR1RowsPerWg = 4;  // rows of one column chunk a lane takes: the column maxima are loaded once
constexpr int kR1Cols = kRank1Threads * 8;        // columns of a chunk at most
struct RowShape {
    uint32_t width;          // columns of a chunk, a multiple of 128
    uint32_t lanes, magic;   // lanes that share a row: width / 8; floor(2^32 / lanes) + 1
    uint32_t groups;         // rows side by side
};
constexpr int kRowHalf = kGroup / 2;

// Where a lane works: columns [c, c + 4) and [c + 64, c + 68), where the tensor has them, of rows r0 + t * groups.  A lane without work
// and a run or row past the tensor's end load from a place that is there (c, c2, the last row): no branch between a wave's loads.
struct RowLane {
    int64_t c, c2, r0;
    bool live, second;
};

// ONE: one row at a time (groups = 1), so that rows and their statistics are the workgroup's, in scalar registers.
template <bool ONE>
__device__ __forceinline__ RowLane row_lane(const RowShape &sh, int64_t C)
{
    RowLane q;
    const uint32_t g = ONE ? 0u : __umulhi(threadIdx.x, sh.magic), l = threadIdx.x - g * sh.lanes;
    q.c = (int64_t)blockIdx.x * sh.width + (l >> 4) * kGroup + (l & 15u) * 4;
    q.r0 = (int64_t)blockIdx.y * ((ONE ? 1u : sh.groups) * kR1RowsPerWg) + g;
    q.live = (ONE ? l < sh.lanes : g < sh.groups) && q.c < C;
    q.second = q.live && q.c + kRowHalf < C;
    q.c = q.live ? q.c : 0;
    q.c2 = q.second ? q.c + kRowHalf : q.c;
    return q;
}

template <bool ONE>
__device__ __forceinline__ int64_t row_of(const RowLane &q, const RowShape &sh, int t)
{
    return q.r0 + (ONE ? t : t * (int)sh.groups);
}

// ---- flat -------------------------------------------------------------------------------
struct FlatCols {
    double inv;         // 1 / C
    uint32_t c, magic;  // C, floor(2^32 / C)
};

// Row and column of the tile's first value b0, from a rounded product with 1 / C and one correction (b0 < 2^44, so the product
// is off by less than one).
__device__ __forceinline__ void flat_base(int64_t b0, const FlatCols &f, int64_t &r0, uint32_t &c0)
{
    int64_t r = (int64_t)((double)b0 * f.inv);
    int64_t c = b0 - r * f.c;
    if (c < 0) {
        c += f.c;
        --r;
    } else if (c >= f.c) {
        c -= f.c;
        ++r;
    }
    r0 = r;
    c0 = (uint32_t)c;
}

// Row (less the tile's first row) and column of the value `off` past the tile's first.  With magic = floor(2^32 / C) the product's
// upper half is the quotient or one less.
__device__ __forceinline__ void flat_at(uint32_t c0, uint32_t off, const FlatCols &f, uint32_t &r, uint32_t &c)
{
    const uint32_t u = c0 + off;
    r = __umulhi(u, f.magic);
    c = u - r * f.c;
    if (c >= f.c) {
        c -= f.c;
        ++r;
    }
}

constexpr int kFlatT = 4;                            // passes of a workgroup
constexpr int kFlatPass = kRank1Threads * 4;         // values of a pass: a run of 4 for each lane
constexpr int kFlatTile = kFlatT * kFlatPass;        // 16 KB of values
constexpr int kFlatSpanLog2 = 3;                     // 8 tiles make a run of 128 KB (xcd_run_order)

// The scales of a lane's run of four values from `idx` on, min(row, column) statistic each.  RUNS: C is a multiple of
// 4, so that a run lies in one row and its column statistics on a 16-byte boundary.
template <bool RUNS>
struct FlatStats {
    float4 col;
    float row, row1;
    uint32_t left;  // values of the run that lie in the first row
};

template <bool RUNS>
__device__ __forceinline__ FlatStats<RUNS> flat_stats(const float *__restrict__ rowmax, const float *__restrict__ colmax,
                                                      int64_t r0, uint32_t c0, uint32_t off, int64_t idx, int64_t n,
                                                      bool whole, const FlatCols &f)
{
    FlatStats<RUNS> s;
    s.col = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    s.row = s.row1 = 1.0f;
    s.left = 4;
    if (!whole && idx >= n)
        return s;
    uint32_t r, c;
    flat_at(c0, off, f, r, c);
    const float *rp = rowmax + r0 + r;
    s.row = s.row1 = rp[0];
    if (RUNS) {
        s.col = *reinterpret_cast<const float4 *>(colmax + c);
        return s;
    }
    s.left = f.c - c;
    const uint32_t wrap1 = c + 1 >= f.c ? f.c : 0u, wrap2 = c + 2 >= f.c ? f.c : 0u, wrap3 = c + 3 >= f.c ? f.c : 0u;
    s.col = make_float4(colmax[c], colmax[c + 1 - wrap1], colmax[c + 2 - wrap2], colmax[c + 3 - wrap3]);
    if (s.left < 4 && (whole || idx + s.left < n))
        s.row1 = rp[1];
    return s;
}

template <bool RUNS>
__device__ __forceinline__ void flat_scales(const FlatStats<RUNS> &s, float *scale)
{
    const float col[4] = {s.col.x, s.col.y, s.col.z, s.col.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float row = (RUNS || (uint32_t)k < s.left) ? s.row : s.row1;
        scale[k] = (col[k] < row) ? col[k] : row;
    }
}

// The tile of a workgroup; base: the operand of four bytes a value.
__device__ __forceinline__ uint32_t flat_tile(const void *base)
{
    return xcd_run_order<kFlatSpanLog2>(blockIdx.x, gridDim.x, run_phase<kFlatSpanLog2>(base, kFlatTile * sizeof(float)));
}

// whole: all of the tile's values are there.  Values past the tensor's end read as zeros.
template <bool RUNS>
__device__ __forceinline__ void flat_load(const float *__restrict__ x, int64_t b0, int64_t n, bool whole, float4 (&a)[kFlatT])
{
#pragma unroll
    for (int t = 0; t < kFlatT; ++t) {
        const int64_t idx = b0 + t * kFlatPass + threadIdx.x * 4;
        if (!whole)
            a[t] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (whole || idx + 4 <= n) {
            a[t] = load4(x + idx);
        } else if (!RUNS && idx < n) {
            a[t].x = x[idx];
            a[t].y = idx + 1 < n ? x[idx + 1] : 0.0f;
            a[t].z = idx + 2 < n ? x[idx + 2] : 0.0f;
        }
    }
}

template <bool RUNS>
__device__ __forceinline__ void flat_stats_of_tile(const float *__restrict__ rowmax, const float *__restrict__ colmax, int64_t b0,
                                                   int64_t n, bool whole, const FlatCols &f, FlatStats<RUNS> (&st)[kFlatT])
{
    int64_t r0;
    uint32_t c0;
    flat_base(b0, f, r0, c0);
#pragma unroll
    for (int t = 0; t < kFlatT; ++t) {
        const uint32_t off = t * kFlatPass + threadIdx.x * 4;
        st[t] = flat_stats<RUNS>(rowmax, colmax, r0, c0, off, b0 + off, n, whole, f);
    }
}

template <bool RUNS>
__device__ __forceinline__ void flat_store(float *__restrict__ out, int64_t idx, int64_t n, bool whole, const float *v)
{
    if (whole || idx + 4 <= n) {
        store4(out + idx, make_float4(v[0], v[1], v[2], v[3]));
    } else if (!RUNS && idx < n) {
        out[idx] = v[0];
        if (idx + 1 < n)
            out[idx + 1] = v[1];
        if (idx + 2 < n)
            out[idx + 2] = v[2];
    }
}

// ---- host: which split, and its shape ----------------------------------------------------
// The rows split where it is the faster one (the table above), and the column groups of its chunks.  Chunks of 16 or 8 groups, whose
// workgroups take runs of 8 or 4 KB, where at most 3 % of them lie beyond the row's end; else narrow ones from 4096 columns on,
// several rows side by side, if rows start on cache lines.  Otherwise a quantiser takes the widest chunk that leaves at most a
// tenth of the lanes idle, else the one that leaves fewest; a dequantiser, which has nothing to keep over the rows but cuts lines
// at a chunk's end, whole rows of 1, 2 or 4 groups, pairs of groups from 12 groups on, and for the rest the flat split.
// Dequantisers (us, 4 / 8 bits; "lanes": with the quantiser's rule for every column count that is a multiple of 128; "before" as
// above; 1.5 to 2 % slower than before: 1280, 1536 and 1920 columns at 4 bits):
//                  lanes         here          before
//   70000 x 1152   82.1 / 74.8   70.7 / 70.6   73.1 / 75.0
//   50000 x 1664   77.1 / 75.0   74.4 / 75.0   73.9 / 76.6
//   36000 x 2176   86.1 / 80.7   72.0 / 74.2   105.9 / 115.8
//   36000 x 2304   77.4 / 75.6   71.5 / 72.4   103.9 / 117.0
//   20000 x 4224   93.4 / 90.0   81.4 / 74.7   81.6 / 81.7
//   15000 x 5504   82.5 / 78.1   79.0 / 75.0   79.3 / 78.4
//   7200 x 11008   72.4 / 72.1   72.4 / 72.2   80.3 / 83.9
// Quantisers: 20000 x 4224 63.0 / 71.5, 59.9 / 68.3, 64.0 / 70.3; 15000 x 5504 60.4 / 67.4, 59.1 / 66.7, 59.3 / 66.4.
inline int64_t row_chunk_groups(int64_t cols, bool quantise)
{
    const int64_t groups = (cols + kGroup - 1) / kGroup;
    for (int64_t wide = 16; wide >= 8; wide /= 2)
        if ((double)cols >= 0.97 * (double)((groups + wide - 1) / wide * wide * kGroup))
            return wide;
    if (cols >= 4096 && cols % kGroup == 0)
        return quantise ? 4 : 2;
    if (!quantise)
        return groups == 1 || groups == 2 || groups == 4 ? groups : groups >= 12 && groups % 2 == 0 ? 2 : 0;
    const int64_t least = (cols + kR1Cols - 1) / kR1Cols;
    double best = 0.0;
    int64_t found = 0;
    for (int64_t k = least; k <= 2 * least + 2 && best < 0.9; ++k) {
        const int64_t wide = (groups + k - 1) / k, lanes = 16 * wide;
        const double use = (double)(kRank1Threads / lanes * lanes) / kRank1Threads * (double)cols / (double)(kGroup * wide * k);
        if (use > best + 0.02) {
            best = use;
            found = wide;
        }
    }
    return found;
}

inline bool rank1_rows(const void *x, const void *colmax, const void *codes, int64_t rows, int64_t cols, bool quantise, RowShape &sh,
                       dim3 &grid)
{
    if (quantise ? cols % kGroup != 0 && cols < 256 : cols % kGroup != 0)
        return false;
    if (cols % 4 != 0 || !aligned_to(x, 16) || !aligned_to(colmax, 16) || !aligned_to(codes, 4))
        return false;
    const int64_t wide = row_chunk_groups(cols, quantise);
    if (wide == 0)
        return false;
    const int64_t chunks = (cols + wide * kGroup - 1) / (wide * kGroup);
    sh.lanes = (uint32_t)(16 * wide);
    sh.width = 8 * sh.lanes;
    sh.magic = (uint32_t)((1ULL << 32) / sh.lanes) + 1u;
    sh.groups = kRank1Threads / sh.lanes;
    const int64_t gy = (rows + (int64_t)sh.groups * kR1RowsPerWg - 1) / ((int64_t)sh.groups * kR1RowsPerWg);
    grid = dim3((uint32_t)chunks, (uint32_t)gy);
    return gy <= 65535 && chunks <= 0x7fffffffLL;
}

// The flat split: columns that an index of 32 bits reaches past a tile, runs on 16-byte boundaries.
inline bool rank1_flat_ok(const void *x, const void *colmax, const void *codes, int64_t cols)
{
    return cols >= 4 && cols <= 0x40000000LL && aligned_to(x, 16) && aligned_to(codes, 4) && (cols % 4 != 0 || aligned_to(colmax, 16));
}

inline FlatCols flat_cols(int64_t cols)
{
    return {1.0 / (double)cols, (uint32_t)cols, (uint32_t)((1ULL << 32) / (uint64_t)cols)};
}

}  // namespace lpmm
