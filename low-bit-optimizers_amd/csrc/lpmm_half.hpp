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

// Larger and smaller of two halfs each, a NaN left out as by fmaxf.  (The compiler's own maximum canonicalises both
// operands first; these come from a conversion and are canonical.)
__device__ __forceinline__ v2h max2(v2h a, v2h b)
{
    v2h r;
    asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

__device__ __forceinline__ v2h min2(v2h a, v2h b)
{
    v2h r;
    asm("v_pk_min_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// largest of a lane's eight values and zero; ABS: of their magnitudes (otherwise no value is negative)
template <bool ABS>
__device__ __forceinline__ float max8(const v2h (&x)[kPairs])
{
    const v2h a = ABS ? max2(abs2(x[0]), abs2(x[1])) : max2(x[0], x[1]);
    const v2h b = ABS ? max2(abs2(x[2]), abs2(x[3])) : max2(x[2], x[3]);
    const v2h r = max2(a, b);
    uint32_t top;  // of the two halfs, in the lower half
    asm("v_max_f16_sdwa %0, %1, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1" : "=v"(top) : "v"(r));
    return fmaxf((float)__builtin_bit_cast(v2h, top).x, 0.0f);
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

// The correctly rounded root of a half from 0 to infinity: on gfx950 the hardware's half root, for every one of them (all are compared
// by the tests).  Elsewhere (ARCH of the Makefile) the float root rounded to half, which may be 1 ulp off: the root of a half lies at
// least 0.5 ulp of a float away from a tie.
__device__ __forceinline__ h16 half_root(h16 x)
{
#if defined(__gfx950__)
    return (h16)__builtin_amdgcn_sqrth(x);
#else
    return (h16)__builtin_amdgcn_sqrtf((float)x);
#endif
}

// The parameter of two elements from their updated moments.  IEEE: divisions as the
// compiler writes them, for kernels that arithmetic does not bound: infinite second moments (with beta2 = 0.999
// gradients above 8090, where (1 - beta2) g^2 passes 65504) divide as in the chain too.
template <bool ZERO, bool IEEE>
__device__ __forceinline__ v2h half_param(v2h p, v2h m, v2h v, const NfHyper &h, const MixConst &c)
{
    const v2h pi = round2(mix_mul(p.x, h.decay, c), mix_mul(p.y, h.decay, c));
    v2h d = {half_root(v.x), half_root(v.y)};
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

// Are a step's constants the usual ones: a lerp weight below 0.5 and an eps that is positive as a half, which keeps every
// denominator positive (rounding is monotonic)?  Known on the host.
__host__ __device__ __forceinline__ bool half_near(float w1) { return fabsf(w1) < 0.5f; }
__host__ __device__ __forceinline__ bool half_eps_positive(float eps) { return eps > 0x1p-25f; }

// A lane's eight elements through the chain; p, m and v are updated in place.  Both branches are uniform.
// OPS: the second moment as the device ops leave it (half_second_moment_ops).  USUAL: the caller knows that the step's constants
// are; without the branches the products and sums of the whole chain read their half operands directly (behind one the compiler
// converts each gradient and first moment for both sides: 2 instructions a value)
template <bool IEEE = false, bool OPS = false, bool USUAL = false>
__device__ __forceinline__ void half_elts8(v2h (&p)[kPairs], const v2h (&g)[kPairs], v2h (&m)[kPairs], v2h (&v)[kPairs],
                                           const NfHyper &h, const MixConst &c, const RoundOnce &once = {})
{
    if (USUAL || half_near(h.w1)) {
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
    if (IEEE || USUAL || half_eps_positive(h.eps)) {
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
    // (mix_mul; written out because the compiler widens x first where another block uses it as well)
    float a, b;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(a) : "v"(x), "v"(rcx), "v"(c.neg_zero));
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(b) : "v"(x), "v"(rcy), "v"(c.neg_zero));
    return round2(a, b);
}

// LDS of the kernels whose normalised values are halfs (bytes): the two maps, then three tables of 256 entries.
//   pairs of the first map, floats: entry b = values of the two codes in byte b;
//   pairs of the second map, as halfs: for the standard map, whose values k / 16 are halfs;
//   the first moment's codes by the upper byte of a half's bits (kEncHalfM), pairs of words.
// One read decodes two codes, at the price of bank conflicts that these kernels, bound by their arithmetic, do not notice.
constexpr uint32_t kHalfPairsM = 128, kHalfPairsV = kHalfPairsM + 2048, kHalfEnc = kHalfPairsV + 1024;
constexpr uint32_t kHalfLdsBytes = kHalfEnc + 2048;

// By 256 threads, in two halves like lds_fill_load and lds_fill_store; the caller synchronises.
struct HalfLdsFill {
    float q;
    float2 m;
    v2h v;
    uint2 enc;
};

__device__ __forceinline__ HalfLdsFill half_lds_load(const float *__restrict__ qmap_m, const float *__restrict__ qmap_v)
{
    const uint32_t t = threadIdx.x;
    HalfLdsFill f;
    f.q = ((t & 16) == 0 ? qmap_m : qmap_v)[t & 15];
    f.m = make_float2(qmap_m[t & 15], qmap_m[t >> 4]);
    f.v = v2h{(h16)qmap_v[t & 15], (h16)qmap_v[t >> 4]};
    f.enc = *reinterpret_cast<const uint2 *>(kEncHalfM[t]);
    return f;
}

__device__ __forceinline__ void half_lds_store(uint32_t *lds, const HalfLdsFill &f)
{
    const uint32_t t = threadIdx.x;
    char *const at = reinterpret_cast<char *>(lds);
    lds[t & 31] = __float_as_uint(f.q);
    *reinterpret_cast<float2 *>(at + kHalfPairsM + 8 * t) = f.m;
    *reinterpret_cast<v2h *>(at + kHalfPairsV + 4 * t) = f.v;
    *reinterpret_cast<uint2 *>(at + kHalfEnc + 8 * t) = f.enc;
}

__device__ __forceinline__ void half_lds_fill(uint32_t *lds, const float *__restrict__ qmap_m, const float *__restrict__ qmap_v)
{
    half_lds_store(lds, half_lds_load(qmap_m, qmap_v));
}
static_assert(kThreads == 256 && kLdsQ0 == 0 && kLdsQ1 == 64, "half_lds_store writes one entry a thread and the maps back to back");

__device__ __forceinline__ uint32_t code_byte(uint32_t w, int j) { return (w >> (8 * j)) & 0xffu; }

// rh(map value * scale) of a lane's eight codes; byte j of w: the codes of pair j
__device__ __forceinline__ void half_decode_m(const uint32_t *lds, uint32_t w, float scale, v2h (&m)[kPairs])
{
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
        const float2 q = lds_read<float2>(lds, kHalfPairsM + 8 * code_byte(w, j));
        m[j] = round2(q.x * scale, q.y * scale);
    }
}

// The same for the second moment.  A product of two halfs is exact as a float, so one rounding to half follows either way and
// the packed product of halfs is that result: where the map's values are halfs.
__device__ __forceinline__ void half_decode_v(const uint32_t *lds, int kind, uint32_t w, const v2h (&scale)[kPairs], v2h (&v)[kPairs],
                                              const MixConst &c)
{
    if (kind == kMapStdV) {
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            v[j] = scale[j] * lds_read<v2h>(lds, kHalfPairsV + 4 * code_byte(w, j));
        return;
    }
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
        const uint32_t b = code_byte(w, j);
        v[j] = round2(mix_mul(scale[j].x, lds_read<float>(lds, kLdsQ1 + 4 * (b & 15u)), c),
                      mix_mul(scale[j].y, lds_read<float>(lds, kLdsQ1 + 4 * (b >> 4)), c));
    }
}

// bytes of two words (codes of the lane's eight values, four a word) -> nibbles
__device__ __forceinline__ uint32_t pack_code_bytes(uint32_t lo, uint32_t hi)
{
    return __builtin_amdgcn_perm(hi | (hi >> 4), lo | (lo >> 4), 0x06040200u);
}

// Codes of eight halfs with the standard first-moment map; any half, a (quiet) NaN gives 15.  A value's bucket is the upper byte of
// its bits, its code the upper half of one multiply-add.
__device__ __forceinline__ uint32_t encode8_half_m(const uint32_t *lds, const v2h (&x)[kPairs])
{
    uint32_t r[kEltsPerLane];
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, x[j]);
        const uint2 a = lds_read<uint2>(lds, kHalfEnc + 8 * ((bits >> 8) & 0xffu)), b = lds_read<uint2>(lds, kHalfEnc + 8 * (bits >> 24));
        asm("v_mad_i32_i16 %0, %1, %2, %3" : "=v"(r[2 * j]) : "v"(bits), "v"(a.y), "v"(a.x));
        asm("v_mad_i32_i16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(r[2 * j + 1]) : "v"(bits), "v"(b.y), "v"(b.x));
    }
    uint32_t w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)  // byte 2 of each
        w[h] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(r[4 * h + 3], r[4 * h + 2], 0x06020c0cu),
                                     __builtin_amdgcn_perm(r[4 * h + 1], r[4 * h], 0x0c0c0602u), 0x07060100u);
    return pack_code_bytes(w[0], w[1]);
}

// Codes of eight halfs in [0, 1] with the standard second-moment map (NaN, negative: 0).  Its midpoints are (k + 0.5) / 16, so the
// code is 16 x rounded to an integer, ties down, less one.  1023 + 16 x, rounded once to a half, is an integer (halfs from 1024 on
// are); with the factor 16 (1 - 2^-11), itself a half, a tie falls below its midpoint, and the next half above, larger by more
// than 2^-11 of its value, does not.  All halfs of the range are compared with the search by the tests.
__device__ __forceinline__ uint32_t encode8_half_v(const v2h (&x)[kPairs])
{
    const v2h factor = {(h16)15.9921875f, (h16)15.9921875f}, offset = {(h16)1023.0f, (h16)1023.0f}, least = {(h16)1024.0f, (h16)1024.0f};
    uint32_t r[kPairs];
#pragma unroll
    for (int j = 0; j < kPairs; ++j)
        r[j] = __builtin_bit_cast(uint32_t, max2(__builtin_elementwise_fma(x[j], factor, offset), least));
    // 1024 + code has the code in its lowest byte
    return pack_code_bytes(__builtin_amdgcn_perm(r[1], r[0], 0x06040200u), __builtin_amdgcn_perm(r[3], r[2], 0x06040200u));
}

// Codes of normalised halfs; any values, a NaN gives 15.
__device__ __forceinline__ uint32_t encode8_half(const uint32_t *lds, uint32_t lds_map, int kind, const v2h (&x)[kPairs])
{
    if (kind == kMapStdM)
        return encode8_half_m(lds, x);
    if (kind == kMapStdV) {
        v2h y[kPairs];  // at most 1, NaNs 1 as well: code 15
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            y[j] = min2(x[j], v2h{(h16)1.0f, (h16)1.0f});
        return encode8_half_v(y);
    }
    // any ascending map: the midpoints below a value, one midpoint at a time (all of them at once would cost the kernels a wave)
    uint32_t codes[kEltsPerLane] = {};
    const float *const q = reinterpret_cast<const float *>(lds) + lds_map / 4;
#pragma unroll 1
    for (int m = 0; m < 15; ++m) {
        const float mid = (q[m] + q[m + 1]) * 0.5f;
#pragma unroll
        for (int k = 0; k < kEltsPerLane; ++k)
            codes[k] += mid < (float)x[k >> 1][k & 1] ? 1u : 0u;
    }
    uint32_t w = 0;
#pragma unroll
    for (int k = 0; k < kEltsPerLane; ++k) {
        const h16 v = x[k >> 1][k & 1];
        w |= (v == v ? codes[k] : 15u) << (4 * k);
    }
    return w;
}

// Codes of rh(v / scale) for a lane's 8 values; |v| <= scale wherever the scale is finite and
// positive (it is a maximum over the values it divides).
__device__ __forceinline__ uint32_t encode8_scaled_h(const uint32_t *lds, uint32_t lds_map, int kind,
                                                     const v2h (&v)[kPairs], float scale, const MixConst &c)
{
    v2h q[kPairs];
    if (kind != kMapGeneric && rc_safe(scale)) {
        // quotients in [-1, 1]
        const float rc = rcp_exact(scale);
#pragma unroll
        for (int j = 0; j < kPairs; ++j)
            q[j] = half_quotients(v[j], rc, rc, c);
        return kind == kMapStdM ? encode8_half_m(lds, q) : encode8_half_v(q);
    }
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
        v2h x = v[j];
        asm volatile("" : "+v"(x));  // what only this branch needs stays in it
        q[j] = v2h{(h16)rh((float)x.x / scale), (h16)rh((float)x.y / scale)};
    }
    return encode8_half(lds, lds_map, kind, q);
}

// (co < ro) ? co : ro for two columns' statistics: non-negative halfs, or NaN for the row.  A NaN column gives the row's
// statistic: rank1_columns makes it infinite beforehand.  A NaN row statistic is the result, as of the packed minimum that hands NaNs on.
__device__ __forceinline__ v2h rank1_columns(v2h co)
{
    const v2h inf = {(h16)__builtin_inff(), (h16)__builtin_inff()};
    return min2_bits(co, inf);
}
__device__ __forceinline__ v2h rank1_scales(v2h co, h16 ro)
{
    const v2h rows = {ro, ro};
    return __builtin_elementwise_minimum(co, rows);
}

}  // namespace lpmm
