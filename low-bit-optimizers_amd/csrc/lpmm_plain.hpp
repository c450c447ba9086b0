// Tensors with fp32 states as part of a launch: records, tiles and checks of what fused_adamw.hip launches alone or beside quantised
// tensors, nonfused_rank1.hip beside the clearing before its first pass and factored.hip beside the end of its statistics; and either
// arithmetic.
#pragma once
#include "lpmm_update.hpp"

#include <string.h>

namespace lpmm {

constexpr int kPlainThreads = 256;

struct FusedArith {
    // code buffers hold exactly ceil(n/2) bytes; a last odd element leaves its high nibble 0
    static constexpr bool kPadded = false;
    Hyper h;
    template <class M, class T>
    __device__ __forceinline__ FusedArith(const M &a, const T &t)
    {
        h.beta1 = a.s[0];
        h.beta2 = a.s[1];
        h.omb1 = a.s[2];
        h.omb2 = a.s[3];
        h.lr = a.s[4];
        h.wd = a.s[5];
        h.eps = a.s[6];
        h.c1 = t.k[0];   // 1 - beta1^step
        h.c2s = t.k[1];  // sqrt(1 - beta2^step)
        h.rc2s = t.k[2]; // 1 / c2s, correctly rounded (host division)
    }
    __device__ __forceinline__ void elt(float &p, float g, float &m, float &v) const { p = adamw_elt(p, g, m, v, h); }
    // per-tensor scalars of a tensor at step `step`, as the reference computes them per thread
    static void per_tensor(float beta1, float beta2, float eps, float step, float (&k)[4])
    {
        bias_corrections(beta1, beta2, step, &k[0], &k[1]);
        k[2] = 1.0f / k[1];
        k[3] = 0.0f;
    }
};

struct NonFusedArith {
    // code buffers are padded to whole tiles plus one byte, as the reference's packing
    // operator lays them out: every nibble of an existing group is written, groups past the
    // tensor hold the code of 0.0
    static constexpr bool kPadded = true;
    NfHyper h;
    template <class M, class T>
    __device__ __forceinline__ NonFusedArith(const M &a, const T &t)
    {
        h.decay = a.s[0];
        h.w1 = a.s[1];
        h.b2 = a.s[2];
        h.w2 = a.s[3];
        h.eps = a.s[4];
        h.neg_step_size = t.k[0];
        h.bc2_sqrt = t.k[1];
        h.rbc2_sqrt = t.k[2];
    }
    __device__ __forceinline__ void elt(float &p, float g, float &m, float &v) const { nonfused_elt(p, g, m, v, h); }
    // per-tensor scalars at step `step`
    static void per_tensor(double beta1, double beta2, double lr, double weight_decay, double eps, double step, float (&k)[4])
    {
        const NfHyper h = make_nf_hyper(beta1, beta2, lr, weight_decay, eps, step);
        k[0] = h.neg_step_size;
        k[1] = h.bc2_sqrt;
        k[2] = h.rbc2_sqrt;
        k[3] = 0.0f;
    }
};

// Tensors with fp32 states that go with the launches of a call; `next`: the first that has not gone yet.
struct PlainSet {
    const lpmm_adamw_fp32_tensor *tensors;
    int64_t count, next;
};

struct TensorF {
    float *p;
    const float *g;
    float *m;
    float *v;
    int64_t n;
    float k[4];  // per-tensor scalars, as in Tensor4
};

constexpr int kMultiFMax = 64;
constexpr int kTileF = 1024;  // 256 threads x 4 elements

struct MultiF {
    TensorF t[kMultiFMax];
    uint32_t tile_start[kMultiFMax + 1];
    int count;
    float s[7];
};

static_assert(sizeof(MultiF) <= 4096, "kernel arguments exceed 4 KB");

// fp32 states, either arithmetic (the FusedArith / NonFusedArith constructors only read the
// scalars, which Multi4 and MultiF name alike)
template <class Arith>
__device__ __forceinline__ void tile_fp32(const MultiF &args, uint32_t tile)
{
    int lo = 0, hi = args.count;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (args.tile_start[mid] <= tile)
            lo = mid;
        else
            hi = mid;
    }
    const TensorF &t = args.t[lo];
    const Arith h(args, t);
    const int64_t tile0 = (int64_t)(tile - args.tile_start[lo]) * kTileF;
#pragma unroll
    for (int k = 0; k < kTileF / kPlainThreads; ++k) {
        const int64_t i = tile0 + k * kPlainThreads + threadIdx.x;
        if (i < t.n) {
            float p = t.p[i], m = t.m[i], v = t.v[i];
            h.elt(p, t.g[i], m, v);
            t.p[i] = p;
            t.m[i] = m;
            t.v[i] = v;
        }
    }
}

inline int check_fp32(const lpmm_adamw_fp32_tensor *tensors, int64_t count, uintptr_t elt_align)
{
    LPMM_REQUIRE_PTR(tensors);
    for (int64_t i = 0; i < count; ++i) {
        const lpmm_adamw_fp32_tensor &t = tensors[i];
        if (t.n < 0 || (t.n + kTileF - 1) / kTileF > 0x7fffffffLL)
            return LPMM_ERR_SIZE;
        if (t.n == 0)
            continue;
        LPMM_REQUIRE_PTR(t.p);
        LPMM_REQUIRE_PTR(t.g);
        LPMM_REQUIRE_PTR(t.m);
        LPMM_REQUIRE_PTR(t.v);
        LPMM_REQUIRE_ALIGN(t.p, elt_align);
        LPMM_REQUIRE_ALIGN(t.g, elt_align);
        LPMM_REQUIRE_ALIGN(t.m, elt_align);
        LPMM_REQUIRE_ALIGN(t.v, elt_align);
    }
    return LPMM_OK;
}

// One launch's records from tensors[i] on, at most kMultiFMax that are not empty: its tiles (0: none left).
template <class PerTensor>
inline uint32_t fill_fp32(MultiF &args, const lpmm_adamw_fp32_tensor *tensors, int64_t count, int64_t &i, PerTensor per_tensor)
{
    int k = 0;
    uint64_t tiles = 0;
    float step = 0.0f;
    args.tile_start[0] = 0;
    while (i < count && k < kMultiFMax) {
        const lpmm_adamw_fp32_tensor &t = tensors[i];
        if (t.n == 0) {
            ++i;
            continue;
        }
        const uint64_t nt = (uint64_t)((t.n + kTileF - 1) / kTileF);
        if (tiles + nt > 0x7fffffffULL)
            break;
        TensorF &d = args.t[k];
        d.p = t.p;
        d.g = t.g;
        d.m = t.m;
        d.v = t.v;
        d.n = t.n;
        if (k != 0 && t.step == step)  // two powers a tensor, 0.1 us, for what tensors of one group share
            memcpy(d.k, args.t[k - 1].k, sizeof d.k);
        else
            per_tensor(step = t.step, d.k);
        tiles += nt;
        args.tile_start[++k] = (uint32_t)tiles;
        ++i;
    }
    args.count = k;
    for (int j = k + 1; j <= kMultiFMax; ++j)
        args.tile_start[j] = (uint32_t)tiles;
    return (uint32_t)tiles;
}

}  // namespace lpmm
