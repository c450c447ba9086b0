// Shared by the two-pass rank-1 step kernels (nonfused_rank1.hip: 4-bit states, the tuned passes;
// nonfused_rank1_bits.hip: 5-8-bit states; nonfused_rank1_ragged.hip: column counts that are no
// multiple of 128): the tensor records of a launch, the tile geometry and small helpers.
#pragma once
#include "lpmm_update.hpp"

namespace lpmm {

constexpr int kThreads = 256;
constexpr int kEltsPerLane = 8;
constexpr int kDppRows = kThreads / 16;  // 128-column groups a workgroup handles per pass
constexpr int kR1Max = 32;               // tensors per launch
constexpr int kR1Many = 64;              // of small ones, in the kernels of nonfused_rank1.hip
// Tile policy: widest tile (lg of 128-column groups), tensor rows per workgroup (more where one pass
// of a narrow tile covers more), workgroups taken to be resident together.
#ifndef LPMM_R1_LG
#define LPMM_R1_LG 1
#endif
#ifndef LPMM_R1_ROWS
#define LPMM_R1_ROWS 64
#endif
#ifndef LPMM_R1_RESIDENT
#define LPMM_R1_RESIDENT 256
#endif
constexpr int kPolicyLgWide = LPMM_R1_LG;
constexpr uint32_t kPolicyRows = LPMM_R1_ROWS, kPolicyResident = LPMM_R1_RESIDENT;
constexpr uint32_t kPolicyRowsHalf = LPMM_R1_ROWS * 2;  // float16 parameters
constexpr uint32_t kPolicyRowsMost = kPolicyRowsHalf;
static_assert(LPMM_R1_LG >= 1 && LPMM_R1_LG <= 3, "a tile is 256 to 1024 columns wide at most");
constexpr int kMaxLgWide = kPolicyLgWide;   // the LDS column arrays hold 128 << kMaxLgWide columns
constexpr int kMaxWide = 1 << kMaxLgWide;
// Per-column data of a tile lives in LDS, not in registers (occupancy): the current column
// statistics in the unused bytes between the maps and the encode table, further arrays after
// the table.
constexpr uint32_t kColBytes = kMaxWide * kGroup * 4;
constexpr uint32_t kColOld = kLdsQ1 + 64;
static_assert(kColOld + kColBytes <= kEncLdsBegin, "column statistics overlap the encode table");
constexpr uint32_t kColExtra = (kLdsBytes + 15) / 16 * 16;  // first byte after the table
// Column maxima of the tile, one slot of 8 x 16 words (+16 words of skew, so that the DPP rows
// of a wave hit different banks) per column group: word k * 16 + lane16 of a slot is element k
// of lane lane16.
constexpr uint32_t kRedSlotWords = kGroup + 16;

// A workgroup covers tile_rows rows x (128 << lg_wide) columns: per pass, (16 >> lg_wide) rows of
// (1 << lg_wide) adjacent groups each.
struct TileShape {
    uint32_t lg_wide : 4;
    uint32_t drop_nan : 4;    // kernels with folded rows: column maxima leave NaNs out, as those of the kernels for any column count do
    uint32_t tile_rows : 24;  // max(the policy's rows, rows of one pass)
    uint32_t comb;            // row blocks whose passes interleave
};

struct TensorR1 {
    float *p;
    const float *g;
    uint8_t *mc;  // fp32 first moment: the moment itself (float[rows * cols]), ms unused
    float *ms;
    float *ms_new;  // first-moment groups wider than 128 values: the scales of the new first moment
    uint8_t *vc;
    const float *row_old;
    const float *col_old;
    float *row_new;
    float *col_new;
    int64_t rows;
    uint32_t col_blocks;  // columns / 128
    float neg_step_size, bc2_sqrt, rbc2_sqrt;
    uint32_t m_lg;  // the first moment's group holds 128 << m_lg values
    uint32_t col_tail;  // columns in the last 128-column block (128 unless the column count is ragged)
    TileShape tile;
};

// How the first moment is kept: 4-bit codes in groups of 128 values (re-quantised where it is
// updated), fp32 (read and written as floats), or 4-bit codes in wider groups (256 .. 4096
// values of the flattened tensor: a group spans several DPP rows, tiles and, where the column
// count is not a multiple of the group size, tensor rows.  The update pass only merges the
// groups' maxima into the next scales, the second pass recomputes the moment from g and the old
// codes, bit-identically, and writes its codes -- what both passes do for the second moment).
enum MomentMode { kMCodes128 = 0, kMFloat = 1, kMCodesWide = 2 };

template <int N>
struct MultiR1N {
    static constexpr int kMax = N;
    TensorR1 t[N];
    uint32_t tile_start[N + 1];  // prefix sum of tiles per tensor; unused slots hold the total
    int count;
    float decay, w1, b2, w2, eps;
};
using MultiR1 = MultiR1N<kR1Max>;

static_assert(sizeof(MultiR1) + 3 * sizeof(void *) + 2 * sizeof(int) <= 4096, "kernel arguments exceed 4 KB");
static_assert(sizeof(MultiR1N<kR1Many>) + 2 * sizeof(void *) <= kMostKernargBytes, "kernel arguments exceed 8 KB");
static_assert(kR1Max <= kWave && kR1Many <= kWave, "one tile_start entry per lane");

// tensor of this workgroup (uniform): the number of later tensors whose first tile is not
// after this one
template <int N>
__device__ __forceinline__ int find_tensor(const MultiR1N<N> &args)
{
    const int lane = threadIdx.x & (kWave - 1);
    const bool started = lane + 1 < N && args.tile_start[lane + 1] <= blockIdx.x;
    return __popcll(__ballot(started));
}

__device__ __forceinline__ void unpack8(const float4 &a, const float4 &b, float (&o)[kEltsPerLane])
{
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
    o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
}

// Where a DPP row of this workgroup works: column group `cg` (fixed), rows row0, row0 + step, ...
struct Geometry {
    int64_t row0;
    uint32_t cg, col_tile;
    int step, passes, wide;
};

__device__ __forceinline__ Geometry geometry(const TileShape &ts, uint32_t col_blocks, uint32_t tile, int drow)
{
    Geometry q;
    q.wide = 1 << ts.lg_wide;
    const uint32_t col_tiles = (col_blocks + q.wide - 1) >> ts.lg_wide;
    const uint32_t rb = tile / col_tiles;
    q.col_tile = tile - rb * col_tiles;
    q.cg = q.col_tile * q.wide + (drow & (q.wide - 1));
    const int pass_rows = kDppRows >> ts.lg_wide;
    q.passes = (int)ts.tile_rows / pass_rows;
    // block k of group grp: pass i covers the rows from (grp * passes * comb + i * comb + k) * pass_rows on
    const uint32_t grp = rb / ts.comb, k = rb - grp * ts.comb;
    q.row0 = (int64_t)grp * ts.tile_rows * ts.comb + (int64_t)k * pass_rows + (drow >> ts.lg_wide);
    q.step = pass_rows * (int)ts.comb;
    return q;
}

__device__ __forceinline__ Geometry geometry(const TensorR1 &t, uint32_t tile, int drow)
{
    return geometry(t.tile, t.col_blocks, tile, drow);
}

// Tile order of the kernels whose rows start anywhere: tiles of 256 columns then meet inside cache lines.  The hardware hands
// neighbouring workgroups to different XCDs; here an XCD takes runs of four neighbouring tiles, so that most of these lines are read by
// and put together in one L2.  Steps on six tensors of 4096 x 4100: 541 -> 516 us, fp32 first moment 613 -> 576, 8 bits 605 -> 584; thirty
// of 1000 x 1000: 213 -> 195 (fp32), 222 -> 202 (8 bits).  Runs of 16: 1 % faster on the large ones, 5 % slower on the small ones.
constexpr uint32_t kXcdNeighbours = 4;
__device__ __forceinline__ uint32_t xcd_neighbours(uint32_t index, uint32_t tiles)
{
    constexpr uint32_t kBlock = kXcds * kXcdNeighbours;
    const uint32_t block0 = index / kBlock * kBlock, in = index - block0;
    return block0 + kBlock <= tiles ? block0 + (in % kXcds) * kXcdNeighbours + in / kXcds : index;
}

// Folded rows.  A tensor of R x C values whose C is no multiple of 128 but of 2^t, 2 <= t < 7, is the same memory as the
// row-major matrix of rows of 2^lg C values, lg = 7 - t, which are a multiple of 128: the
// 128-value groups of the first moment, cut from the flattened tensor (lpmm/functional.py:404-422),
// never straddle such a row, so the kernels for whole column blocks apply to that matrix (GPT-2-XL's
// d = 1600 and 3 d = 4800: double rows; 408 columns: rows of sixteen).  Where R is no multiple of 2^lg the last row of the matrix, and
// in it the last group, is a part.  What changes is where a value's statistics sit: value c of a row of the matrix
// lies in tensor row (r << lg) + c / C at column c mod C, and a DPP row's 128 values lie in one or two tensor rows, split at a run of
// four (C is 64 or at least 128).  The record
// keeps the tensor's own shape (col_blocks = ceil(C / 128), col_tail = C - 128 (col_blocks - 1)); kernels instantiated
// with FOLD read it this way, tensors with whole column blocks in the same launch as before.
// Made for tensors of many rows: fewer than 16 rows of the matrix leave its tiles mostly empty (walk.cpp: worth_folding, says which go here).
// The first moment is then written where it is computed, all tiles but the last are full, and one kind of launch serves nearly every model,
// where the kernels for any column count (nonfused_rank1_any.hip) and for multiples of 8 (nonfused_rank1_ragged.hip), which split the
// groups' maxima between rows and write the first moment in the second pass, took 19 bytes a value, launches and new
// code arrays of their own.  Steps in us: 50257 x 1600 345 -> 278, 31426 x 408 71 -> 62, six of 4096 x 4100 460 -> 343, 1000000 x 136 765 ->
// 578, thirty of 88 x 88 x 3 x 3 111 -> 48 (the host in both), sixty of 56 x 56 x 3 x 3 208 -> 69;
// fp32 first moment: 50257 x 1600 363 -> 341, six of 4096 x 4100 499 -> 434, 24 of 200 x 200 60 -> 36;
// 8 bits: 50257 x 1600 370 -> 307, six of 4096 x 4100 524 -> 385, 24 of 200 x 200 87 -> 37; groups of 256: 50257 x 1600
// 337 -> 293, six of 4096 x 4100 456 -> 369.  Double rows keep kernels of their own (whole
// last rows, halves instead of runs): GPT-2-XL's 192 matrices take 4928 us with them, 4962 to 5025 without.
struct Fold {
    uint32_t real_cols, col_blocks;  // columns of the tensor; column blocks of the matrix the kernel works on
    uint32_t lg;
    int64_t rows;                    // rows of that matrix
    int64_t tensor_rows, values;
};

// 7 - t of a column count that folds
__host__ __device__ __forceinline__ uint32_t fold_lg(uint32_t cols) { return 7u - (uint32_t)__builtin_ctz(cols); }

template <bool FOLD>
__device__ __forceinline__ Fold fold_of(const TensorR1 &t)
{
    Fold f;
    f.real_cols = (t.col_blocks - 1) * kGroup + t.col_tail;
    f.lg = FOLD && t.col_tail != (uint32_t)kGroup ? fold_lg(f.real_cols) : 0u;
    f.col_blocks = f.lg != 0 ? f.real_cols >> (7u - f.lg) : t.col_blocks;
    f.tensor_rows = t.rows;
    f.rows = FOLD ? (t.rows + ((int64_t)1 << f.lg) - 1) >> f.lg : t.rows;
    f.values = t.rows * f.real_cols;
    return f;
}

// column of the tensor for column c of the matrix
__device__ __forceinline__ uint32_t fold_col(const Fold &f, uint32_t c) { return f.lg != 0 ? c % f.real_cols : c; }

// Column block cg of the matrix: the first tensor row it lies in, counted within a row of the matrix, and how many of its values do (128
// or more: all).
struct FoldSpan {
    uint32_t first, split;
};
__device__ __forceinline__ FoldSpan fold_span(const Fold &f, uint32_t cg)
{
    FoldSpan s;
    s.first = f.lg != 0 ? cg * kGroup / f.real_cols : 0u;
    s.split = (s.first + 1u) * f.real_cols - cg * kGroup;
    return s;
}

// The one or two tensor rows of a column block in row r of the matrix (of the last ones, where there are none).  No branch: a pass's loads
// of the row statistics stay among its other loads, ahead of the first wait.
__device__ __forceinline__ void fold_rows(const Fold &f, const FoldSpan &s, int64_t r, int64_t &r0, int64_t &r1)
{
    const int64_t last = f.tensor_rows - 1;
    r0 = (r << f.lg) + s.first;
    r1 = r0 + (s.split < (uint32_t)kGroup ? 1 : 0);
    r0 = r0 < last ? r0 : last;
    r1 = r1 < last ? r1 : last;
}

// Double rows: the tensor rows of the two halves of column block cg in row r, half h in the second one where halves[h] is 1.
__device__ __forceinline__ void double_halves(const Fold &f, uint32_t cg, uint32_t (&halves)[2])
{
    halves[0] = f.lg != 0 && cg * kGroup >= f.real_cols ? 1u : 0u;
    halves[1] = f.lg != 0 && cg * kGroup + 64 >= f.real_cols ? 1u : 0u;
}

// Row maxima of a tile.  An atomic maximum on global memory goes out to the fabric (the L2s of
// the XCDs are not coherent with each other), and the passes of a tile produce one per tensor row,
// column group and pass: 0.008 per element, a tenth of the first pass's DRAM transactions together
// with its partial writes.  So the maxima of a tile's rows meet in LDS first -- slot 2 * (row of
// the tile) + (tensor row of a double row) -- and one global atomic per row and
// tile follows the passes, issued by neighbouring threads for neighbouring rows (LLaMA-7B-shaped
// set 21.23 -> 20.85 ms per step, GPT-2-XL-shaped set 6.30 -> 5.71 ms).
constexpr int kRowSlots = 2 * (int)kPolicyRowsMost;
static_assert(kRowSlots <= kThreads, "one thread per row slot");
static_assert(kPolicyRows / 4 >= (uint32_t)kDppRows, "a tile holds the policy's rows: one slot pair per row");

__device__ __forceinline__ int row_slot(const TileShape &ts, int pass, int drow)
{
    return 2 * (pass * (kDppRows >> ts.lg_wide) + (drow >> ts.lg_wide));
}

// after the passes and a barrier: rows = rows of the matrix the tile works on; lg: 1 where they are double rows
__device__ __forceinline__ void flush_row_maxima(const uint32_t *rowred, const TileShape &ts, const Geometry &q, int drow,
                                                 int64_t rows, float *__restrict__ row_new, uint32_t lg = 0)
{
    if (threadIdx.x >= (uint32_t)kRowSlots)
        return;
    const int pr = kDppRows >> ts.lg_wide;
    const int local = threadIdx.x >> 1, half = threadIdx.x & 1;
    const int pass = local / pr, in_pass = local - pass * pr;
    // the first row of the tile's first pass: row0 of this thread's DPP row less its place in the pass
    const int64_t r = (q.row0 - (drow >> ts.lg_wide)) + (int64_t)pass * q.step + in_pass;
    if (pass < q.passes && r < rows && half < (1 << lg))
        atomic_max_nonneg(row_new + (r << lg) + half, __uint_as_float(rowred[threadIdx.x]));
}

// Folded rows other than double ones: four slots a row of the tile, for the up to three tensor rows that 256 columns lie in.
constexpr int kFoldSlots = 4 * (int)kPolicyRowsMost;
__device__ __forceinline__ void flush_row_maxima_fold(const uint32_t *rowred, const TileShape &ts, const Geometry &q, int drow, const Fold &f,
                                                      float *__restrict__ row_new)
{
    const int pr = kDppRows >> ts.lg_wide;
    const uint32_t c0 = q.col_tile * (uint32_t)q.wide * kGroup, first = fold_span(f, q.col_tile * (uint32_t)q.wide).first;
    for (int s = threadIdx.x; s < kFoldSlots; s += kThreads) {
        const int local = s >> 2, pass = local / pr, in_pass = local - pass * pr;
        const uint32_t in = first + (uint32_t)(s & 3);  // of the tensor rows of a row of the matrix
        const int64_t r = (q.row0 - (drow >> ts.lg_wide)) + (int64_t)pass * q.step + in_pass, row = (r << f.lg) + in;
        if (pass < q.passes && r < f.rows && in < (1u << f.lg) && (uint64_t)in * f.real_cols < (uint64_t)c0 + (uint32_t)q.wide * kGroup &&
            row < f.tensor_rows)
            atomic_max_nonneg(row_new + row, __uint_as_float(rowred[s]));
    }
}

// Codes of a plain 0.0 into the padding [n, n_padded) of a packed array and 0 into the extra
// last byte; one workgroup.  n and n_padded are multiples of 8, the array is 4-byte aligned.
__device__ __forceinline__ void write_padding(uint8_t *codes, int64_t n, int64_t n_padded, uint32_t zero_word)
{
    for (int64_t i = n + (int64_t)threadIdx.x * kEltsPerLane; i < n_padded; i += kThreads * kEltsPerLane)
        *reinterpret_cast<uint32_t *>(codes + (i >> 1)) = zero_word;
    if (threadIdx.x == 0)
        codes[n_padded / 2] = 0;
}

// Loads of what the second pass reads again (the gradient, the second moment's codes): without the nontemporal hint (KEEP) where a launch's
// gradients fit the memory-side cache, which then serves the second pass.
template <bool KEEP>
__device__ __forceinline__ float4 load4_for(const float *p)
{
    return KEEP ? *reinterpret_cast<const float4 *>(p) : load4(p);
}
template <bool KEEP>
__device__ __forceinline__ uint32_t load_u16_for(const uint16_t *p) { return KEEP ? *p : load_u16(p); }
template <bool KEEP>
__device__ __forceinline__ uint32_t load_u32_for(const uint32_t *p) { return KEEP ? *p : load_u32(p); }

struct PlainSet;  // lpmm_plain.hpp

// One launch's tensors with the tile shapes of either pass (they differ: pass_rows_policy), and its workgroups.
template <int N>
struct R1LaunchN {
    static constexpr int kMax = N;
    MultiR1N<N> update, requant;
    uint32_t update_tiles, requant_tiles;
    bool keep;  // the update pass leaves what the second pass reads again in the cache
};
using R1Launch = R1LaunchN<kR1Max>;

// The launches of the other kernel families (defined next to their kernels).
void launch_rank1_bits(const R1Launch &l, bool wraps, const float *qmap_m, const float *qmap_v, int bits_m,
                       int bits_v, const uint32_t *table_m, const uint32_t *table_v, hipStream_t stream);
void launch_rank1_ragged(const R1Launch &l, const float *qmap_m, const float *qmap_v, hipStream_t stream);
// any column count and alignment (nonfused_rank1_any.hip)
enum AnyKind : int {
    kAnyCodes4 = LPMM_RANK1_CODES4,
    kAnyFloatM = LPMM_RANK1_FLOAT_M,
    kAnyBits = LPMM_RANK1_CODES8,
    kAnyHalf = LPMM_RANK1_HALF
};
struct NewCodes {  // where the second pass puts a tensor's codes
    uint8_t *m[kR1Max], *v[kR1Max];
    bool runs;  // every tensor of the launch may be taken in runs of four values (rank1_any_runs)
};
static_assert(sizeof(MultiR1) + sizeof(NewCodes) + 6 * sizeof(void *) <= kMostKernargBytes, "kernel arguments exceed 8 KB");
bool rank1_any_runs(const lpmm_rank1_any_tensor &t, AnyKind kind);
// passes: 1 the first, 2 the second, 3 both
void launch_rank1_any(const R1Launch &l, const NewCodes &out, const float *qmap_m, const float *qmap_v,
                      AnyKind kind, int bits_m, int bits_v, const uint32_t *table_m, const uint32_t *table_v, int passes, hipStream_t stream);
// float16 parameters (nonfused_half.hip): p, g, the first moment's scales and the current statistics
// of the records point at halfs, the next statistics at float work arrays
void launch_rank1_half(const R1Launch &l, const float *qmap_m, const float *qmap_v, hipStream_t stream);
// statistics and scale of short vectors (rank1_nd.hip): the checks and the launches of lpmm_rank1_small_fold_scale_multi
int check_small_vectors(const lpmm_rank1_small_vector *vectors, int64_t count);
int launch_small_vectors(const lpmm_rank1_small_vector *const *vectors, int64_t count, hipStream_t stream);
// the records of lpmm_nonfused_adamw_rank1_any_step_multi; float16: the next statistics and scales of the records are
// float work arrays (rank1_any_half sets them up and writes the halfs out)
int rank1_any_step_multi(const lpmm_rank1_any_tensor *tensors, int64_t count, AnyKind kind, uint32_t m_lg, const float *qmap_m,
                         int bits_m, const void *table_m, const float *qmap_v, int bits_v, const void *table_v, double beta1,
                         double beta2, double lr, double weight_decay, double eps, int passes, void *stream,
                         PlainSet *plain = nullptr);
int rank1_any_half(const lpmm_rank1_any_tensor *tensors, int64_t count, const float *qmap_m, const float *qmap_v, double beta1,
                   double beta2, double lr, double weight_decay, double eps, void *stream);
int rank1_step_multi_half(const lpmm_nonfused_rank1_tensor *tensors, int64_t count, const float *qmap_m,
                          const float *qmap_v, double beta1, double beta2, double lr, double weight_decay, double eps,
                          void *stream);

}  // namespace lpmm
