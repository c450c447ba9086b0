// The op chain of the non-fused step on float16 parameters, in registers: shared by nonfused_half.hip
// (the tuned passes) and nonfused_rank1_any.hip (any column count).
#pragma once
#include "rank1_tiles.hpp"

namespace lpmm {

typedef _Float16 h16;
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4h load_h4(const h16 *p) { return __builtin_nontemporal_load(reinterpret_cast<const v4h *>(p)); }

// One rounding to half (nearest even, subnormals kept), as at the end of every op of the chain.  The
// float result is pinned in a register first: otherwise the compiler merges the producing operation
// with the conversion into one mixed-precision instruction (v_fma_mixlo_f16), whose result is rounded
// once, from the exact value, where PyTorch's kernels round the float result a second time -- one
// value in a few thousand then differs in the last place of the half.
__device__ __forceinline__ float rh(float x)
{
    asm("" : "+v"(x));
    return (float)(h16)x;
}

// The chain works on pairs of halfs in one register each: two float results go back to halfs in one
// instruction (v_cvt_pk_f16_f32), and a product or sum takes its half operands out of the pairs by itself
// (v_fma_mix_f32: float arithmetic, one rounding, any operand a half of a register).  The compiler forms
// that instruction from an fma of widened halfs only, so products and sums are written as fma(a, b, -0)
// and fma(a, 1, b) -- exactly a * b and a + b, signs of zeros included -- with the two constants hidden
// from it.  A rounding to half then costs half an instruction instead of two conversions; the update pass
// is bound by its arithmetic.
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef uint16_t v2u __attribute__((ext_vector_type(2)));
constexpr int kPairs = kEltsPerLane / 2;

struct MixConst {
    float one, neg_zero;
};

__device__ __forceinline__ MixConst mix_const()
{
    MixConst c = {1.0f, -0.0f};
    asm("" : "+v"(c.one), "+v"(c.neg_zero));
    return c;
}

__device__ __forceinline__ float mix_mul(h16 a, float b, const MixConst &c) { return __builtin_fmaf((float)a, b, c.neg_zero); }
__device__ __forceinline__ float mix_add(h16 a, float b, const MixConst &c) { return __builtin_fmaf((float)a, c.one, b); }

// a * b + c rounded to half once, from the exact result (v_fma_mixlo_f16: nothing pins the float result here)
__device__ __forceinline__ h16 round_once_fma(float a, float b, h16 c) { return (h16)__builtin_fmaf(a, b, (float)c); }

// rh of two values; see rh for the pins
__device__ __forceinline__ v2h round2(float a, float b)
{
    asm("" : "+v"(a), "+v"(b));
    const v2f t = {a, b};
    return __builtin_convertvector(t, v2h);
}

__device__ __forceinline__ v2h abs2(v2h x)
{
    return __builtin_bit_cast(v2h, __builtin_bit_cast(uint32_t, x) & 0x7fff7fffu);
}

// Larger of two halfs each, a NaN left out as by fmaxf.  (The compiler's own maximum canonicalises both
// operands first; these come from a conversion and are canonical.)
__device__ __forceinline__ v2h max2(v2h a, v2h b)
{
    v2h r;
    asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// largest of a lane's eight values and zero; ABS: of their magnitudes (otherwise no value is negative)
template <bool ABS>
__device__ __forceinline__ float max8(const v2h (&x)[kPairs])
{
    const v2h a = ABS ? max2(abs2(x[0]), abs2(x[1])) : max2(x[0], x[1]);
    const v2h b = ABS ? max2(abs2(x[2]), abs2(x[3])) : max2(x[2], x[3]);
    const v2h r = max2(a, b);
    return fmaxf(fmaxf((float)r.x, (float)r.y), 0.0f);
}

// maxima and minima of non-negative halfs are those of their bit patterns
__device__ __forceinline__ v2h max2_bits(v2h a, v2h b)
{
    return __builtin_bit_cast(v2h, __builtin_elementwise_max(__builtin_bit_cast(v2u, a), __builtin_bit_cast(v2u, b)));
}
__device__ __forceinline__ v2h min2_bits(v2h a, v2h b)
{
    return __builtin_bit_cast(v2h, __builtin_elementwise_min(__builtin_bit_cast(v2u, a), __builtin_bit_cast(v2u, b)));
}

__device__ __forceinline__ void pairs_of(const v4h &a, const v4h &b, v2h (&o)[kPairs])
{
    o[0] = a.xy; o[1] = a.zw; o[2] = b.xy; o[3] = b.zw;
}

// a lane's eight values of a group: four at p, four 64 further on
__device__ __forceinline__ void store_pairs(h16 *p, const v2h (&x)[kPairs])
{
    typedef uint32_t v2w __attribute__((ext_vector_type(2)));
    const v2w lo = {__builtin_bit_cast(uint32_t, x[0]), __builtin_bit_cast(uint32_t, x[1])};
    const v2w hi = {__builtin_bit_cast(uint32_t, x[2]), __builtin_bit_cast(uint32_t, x[3])};
    __builtin_nontemporal_store(lo, reinterpret_cast<v2w *>(p));
    __builtin_nontemporal_store(hi, reinterpret_cast<v2w *>(p + 64));
}

// v.mul_(beta2).addcmul_(g, g, value=1 - beta2) on half tensors, as PyTorch's CPU kernel: v + (value * g) * g
__device__ __forceinline__ v2h half_second_moment(v2h v, v2h g, const NfHyper &h, const MixConst &c)
{
    v = round2(mix_mul(v.x, h.b2, c), mix_mul(v.y, h.b2, c));
    const float ax = mix_mul(g.x, mix_mul(g.x, h.w2, c), c), ay = mix_mul(g.y, mix_mul(g.y, h.w2, c), c);
    return round2(mix_add(v.x, ax, c), mix_add(v.y, ay, c));
}

// The same as PyTorch's GPU kernels leave it, for the kernels that stand for the chain of device ops (any column
// count, states that are not quantised): v + value * (g * g), the square exact in float.  Each of the two ops, the product by
// beta2 and this sum, rounds twice (to float, then to half) in whole blocks of 2048 values if all its operands lie on 16-byte
// boundaries, and once (a mixed-precision fma) behind them and everywhere on other boundaries.  With beta2 = 0.999 one
// gradient in a few hundred puts the sum half way between two halfs, where that shows; a product does in ten thousand.
constexpr int64_t kOpsBlock = 2048;

// how many values of the flattened tensor are rounded twice by an op on these operands
__device__ __forceinline__ int64_t ops_twice(const void *a, const void *b, int64_t n)
{
    return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0 ? n / kOpsBlock * kOpsBlock : 0;
}

// which of a lane's values the product and the sum round once, a bit per value
struct RoundOnce {
    uint32_t product, sum;
};

// pair j of the lane's
__device__ __forceinline__ v2h half_second_moment_ops(v2h v, v2h g, const NfHyper &h, const MixConst &c, const RoundOnce &once, int j)
{
    const h16 none = (h16)c.neg_zero;
    v2h d = round2(mix_mul(v.x, h.b2, c), mix_mul(v.y, h.b2, c));
    if (once.product & (1u << (2 * j)))
        d.x = round_once_fma((float)v.x, h.b2, none);
    if (once.product & (2u << (2 * j)))
        d.y = round_once_fma((float)v.y, h.b2, none);
    const float gx = mix_mul(g.x, (float)g.x, c), gy = mix_mul(g.y, (float)g.y, c);
    v2h r = round2(mix_add(d.x, h.w2 * gx, c), mix_add(d.y, h.w2 * gy, c));
    if (once.sum & (1u << (2 * j)))
        r.x = round_once_fma(h.w2, gx, d.x);
    if (once.sum & (2u << (2 * j)))
        r.y = round_once_fma(h.w2, gy, d.y);
    return r;
}

// m.lerp_(g, 1 - beta1); NEAR: the weight lies below 0.5 (lerp_w)
template <bool NEAR>
__device__ __forceinline__ float half_lerp(h16 m, h16 g, float w, const MixConst &c)
{
    const float d = __builtin_fmaf((float)g, c.one, -(float)m);
    return NEAR ? __builtin_fmaf(w, d, (float)m) : __builtin_fmaf(w - 1.0f, d, (float)g);
}

// x / d, correctly rounded (div_fast).  ZERO: the denominator may be zero: float16 rounds the default eps of
// 1e-8 to zero, so the denominator of an element whose second moment is zero is zero and the parameter
// becomes infinite or NaN, as in the reference; the quotient of the approximate reciprocal is already the
// IEEE result then (x * inf).
template <bool ZERO>
__device__ __forceinline__ float half_quotient(float x, h16 dh)
{
    const float d = (float)dh, rc = __builtin_amdgcn_rcpf(d);
    const float q = x * rc;
    const float r = __builtin_fmaf(-q, d, x);
    const float c = __builtin_fmaf(r, rc, q);
    return ZERO && d == 0.0f ? q : c;
}

// The parameter of two elements from their updated moments.  The root of a half rounded to half lies at
// least 0.5 ulp of a float away from a tie, and the hardware's float root (1 ulp) rounds to the same half as
// the correctly rounded one for every half (all of them are compared by the tests).  IEEE: divisions as the
// compiler writes them, for kernels that arithmetic does not bound: infinite second moments (with beta2 = 0.999
// gradients above 8090, where (1 - beta2) g^2 passes 65504) divide as in the chain too.
template <bool ZERO, bool IEEE>
__device__ __forceinline__ v2h half_param(v2h p, v2h m, v2h v, const NfHyper &h, const MixConst &c)
{
    const v2h pi = round2(mix_mul(p.x, h.decay, c), mix_mul(p.y, h.decay, c));
    v2h d = round2(__builtin_amdgcn_sqrtf((float)v.x), __builtin_amdgcn_sqrtf((float)v.y));
    float q[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // div_by_rc(d, bc2_sqrt, rbc2_sqrt)
        if (IEEE) {
            q[i] = (float)d[i] / h.bc2_sqrt;
            continue;
        }
        q[i] = mix_mul(d[i], h.rbc2_sqrt, c);
        q[i] = __builtin_fmaf(__builtin_fmaf(-q[i], h.bc2_sqrt, (float)d[i]), h.rbc2_sqrt, q[i]);
    }
    d = round2(q[0], q[1]);
    d = round2(mix_add(d.x, h.eps, c), mix_add(d.y, h.eps, c));
    const float nx = mix_mul(m.x, h.neg_step_size, c), ny = mix_mul(m.y, h.neg_step_size, c);
    const float ux = IEEE ? nx / (float)d.x : half_quotient<ZERO>(nx, d.x);
    const float uy = IEEE ? ny / (float)d.y : half_quotient<ZERO>(ny, d.y);
    return round2(mix_add(pi.x, ux, c), mix_add(pi.y, uy, c));
}

// A lane's eight elements through the chain; p, m and v are updated in place.  Both branches are uniform.
// OPS: the second moment as the device ops leave it (half_second_moment_ops)
template <bool IEEE = false, bool OPS = false>
__device__ __forceinline__ void half_elts8(v2h (&p)[kPairs], const v2h (&g)[kPairs], v2h (&m)[kPairs], v2h (&v)[kPairs],
                                           const NfHyper &h, const MixConst &c, const RoundOnce &once = {})
{
    if (fabsf(h.w1) < 0.5f) {
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            m[j] = round2(half_lerp<true>(m[j].x, g[j].x, h.w1, c), half_lerp<true>(m[j].y, g[j].y, h.w1, c));
    } else {
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            m[j] = round2(half_lerp<false>(m[j].x, g[j].x, h.w1, c), half_lerp<false>(m[j].y, g[j].y, h.w1, c));
    }
#pragma unroll
    for (int j = 0; j < kPairs; ++j)
        v[j] = OPS ? half_second_moment_ops(v[j], g[j], h, c, once, j) : half_second_moment(v[j], g[j], h, c);
    // an eps that is positive as a half keeps every denominator positive: rounding is monotonic
    if (IEEE || h.eps > 0x1p-25f) {
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            p[j] = half_param<false, IEEE>(p[j], m[j], v[j], h, c);
    } else {
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            p[j] = half_param<true, IEEE>(p[j], m[j], v[j], h, c);
    }
}

// rh(x / s) of two halfs given rc = RN(1 / s), s in the range in which that is exact, 0 <= |x| <= s: one
// product.  With the significands as integers V, S in [1024, 2047] the quotient's distance from a rounding
// boundary M of halfs (an odd integer below 4096) is |V 2^j - M S| / S >= 1 / S >= 1 / 2047 -- never zero, as
// M would have to divide V -- and the product's error is at most M 2^-23 (1 + 2^-25) < 1 / 2047, so it
// falls on the quotient's side of every boundary.  (Quotients below 2^-14, which have fewer bits as halfs, may
// round otherwise; no map the closed forms serve has a midpoint there.)
__device__ __forceinline__ v2h half_quotients(v2h x, float rcx, float rcy, const MixConst &c)
{
    return round2(mix_mul(x.x, rcx, c), mix_mul(x.y, rcy, c));
}

// Codes of rh(v / scale) for a lane's 8 values; |v| <= scale wherever the scale is finite and
// positive (it is a maximum over the values it divides).
__device__ __forceinline__ uint32_t encode8_scaled_h(const uint32_t *lds, uint32_t lds_map, int kind,
                                                     const v2h (&v)[kPairs], float scale, const MixConst &c)
{
    float x[kEltsPerLane];
    if (kind != kMapGeneric && rc_safe(scale)) {
        // quotients in [-1, 1], no NaN: the closed forms of the standard maps apply as they are
        const float rc = rcp_exact(scale);
#pragma unroll
        for (int j = 0; j < kPairs; ++j) {
            const v2h q = half_quotients(v[j], rc, rc, c);
            x[2 * j] = (float)q.x;
            x[2 * j + 1] = (float)q.y;
        }
        return kind == kMapStdM ? encode8_std_m(lds, x) : encode8_std_v(x);
    }
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
        x[2 * j] = rh((float)v[j].x / scale);
        x[2 * j + 1] = rh((float)v[j].y / scale);
    }
    return encode8_plain(lds, lds_map, kind, x);
}

// (co < ro) ? co : ro for two columns' statistics: non-negative halfs or NaN.  On bit patterns a NaN is the
// largest, so a NaN column gives the row's statistic as the comparison does; a NaN row statistic is the result.
__device__ __forceinline__ v2h rank1_scales(v2h co, h16 ro)
{
    const v2h rows = {ro, ro};
    return ro == ro ? min2_bits(co, rows) : rows;
}

}  // namespace lpmm
