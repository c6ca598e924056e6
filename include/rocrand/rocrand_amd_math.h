// rocrand_amd_math.h -- scalar output transforms of the reference's distributions
// (rocrand_uniform.h, rocrand_normal.h, rocrand_log_normal.h) on gfx950, shared by the
// library's kernels and the device API (rocrand_kernel.h).
//
// Uniforms are bit-exact (exact power-of-two scalings or the reference's own double
// arithmetic).  The Box-Muller angle and the affine steps are evaluated operation by
// operation (no contraction) as the reference host path does; the transcendental
// functions are evaluated in double with short fixed polynomials and rounded once.
#pragma once

#include "rocrand_amd_engines.h"
#include "rocrand_amd_mathtab.h"

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <stdint.h>


namespace rocrand_amd_engine
{

// rocrand_common.h:24-37
constexpr float  R_2POW16_INV     = 1.5258789e-05f;
constexpr float  R_2POW16_INV_2PI = 9.58738e-05f;
constexpr float  R_2POW32_INV     = 2.3283064e-10f;
constexpr double R_2POW32_INV_DBL = 2.3283064365386963e-10;
constexpr double R_2POW64_INV_DBL = 5.4210108624275221700372640043497e-20;
constexpr float  R_2POW32_INV_2PI = 1.46291807e-09f;
constexpr double R_2POW53_INV_DBL = 1.1102230246251565e-16;
constexpr double R_PI_DBL         = 3.1415926535897932;
constexpr float  R_2PI            = 6.2831855f;
constexpr float  R_SQRT2          = 1.4142135f;

// ---------------------------------------------------------------- scalar math
// Float transcendentals evaluated in double and rounded once, written for the
// arguments the transforms produce, with short fixed polynomials instead of the
// general-purpose library routines:
//   neg2log (Box-Muller radius, u a positive normal float in [2^-32, 1]): one table load
//        indexed by u's exponent and 6 leading mantissa bits, |u a - 1| < 2^-7, series to
//        r^4 (relative error < 2^-30) or r^6 (< 2^-44);
//   sin/cos of a Box-Muller angle: table entry from the word that the angle came from,
//        series to a^7 / a^6 on |a| < 0.0124 (relative error < 2^-51, also next to the zeros);
//   exp_acc: reduction by ln2/32 in two parts, 2^(j/32) from rocrand_amd_mathtab.h, series of
//        exp(r) - 1 to r^5 on |r| < 0.0109 (relative error < 2^-48), scaling by 2^e in double.
// The r^6 log, sin/cos and exp round to the correctly rounded float result but next to a
// rounding boundary (relative distance 2^-44 or less), so each differs from the host
// libm's float result by at most the host's own error (< 1 ulp).

// Host and device compile the same code (the tests' host twins check it), with these in
// place of the device's intrinsics; the hardware's reciprocal square roots are good to
// 2^-24 (double) and one ulp (float).
__host__ __device__ __forceinline__ uint32_t rr_float_bits(float x)
{
    uint32_t b;
    __builtin_memcpy(&b, &x, sizeof(b));
    return b;
}
__host__ __device__ __forceinline__ double rr_rsq(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return (double)(float)(1.0 / __builtin_sqrt(x));
#endif
}
__host__ __device__ __forceinline__ float rr_rsqf(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsqf(x);
#else
    return (float)(1.0 / __builtin_sqrt((double)x));
#endif
}

// -2 ln u for a float u in [2^-32, 1]: the exponent and 6 leading mantissa bits index
// rr_bm_logtab (a = 2^-k / c, b = 2 ln a), r = u a - 1 (one rounding-free fused operation)
// and -2 ln u = b - 2 log1p(r), to r^4 or r^6.  u = 1 gives -0, as the reference's
// -2.0f * logf(1.0f).
template<int DEG>
__host__ __device__ __forceinline__ double neg2log(float u)
{
    ROCRAND_AMD_FP_EXACT
    const uint32_t off = ((rr_float_bits(u) >> 17) << 4) - RR_BM_EMIN * 64u * 16u; // entry (exponent, i)
    const double2  t   = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(rr_bm_logtab) + off);
    const double   r   = __builtin_fma((double)u, t.x, -1.0);
    double         p;
    if constexpr(DEG == 4)
        p = __builtin_fma(r, 0.5, -2.0 / 3);
    else
    {
        p = __builtin_fma(r, 1.0 / 3, -2.0 / 5);
        p = __builtin_fma(p, r, 0.5);
        p = __builtin_fma(p, r, -2.0 / 3);
    }
    p = __builtin_fma(p, r, 1.0);
    p = __builtin_fma(p, r, -2.0);
    return __builtin_fma(p, r, t.y);
}

// logf of u, correctly rounded (an exact scaling of neg2log's rounding).
__host__ __device__ __forceinline__ float logf_unit(float u)
{
    return -0.5f * (float)neg2log<6>(u);
}

// sqrtf, correctly rounded, for 0 and floats from 2^-96 up: the hardware reciprocal square
// root, then one step from the exact residual x - s^2 (equal to the correctly rounded root
// for every float of [2^-30, 2^8), checked exhaustively on gfx950; the compiler's sqrtf
// adds a rescaling of tiny inputs and takes twice as many instructions).
__host__ __device__ __forceinline__ float sqrtf_unit(float x)
{
    ROCRAND_AMD_FP_EXACT
    const float y = rr_rsqf(__builtin_fmaxf(x, 0x1p-96f));
    const float s = x * y;
    const float e = __builtin_fmaf(-s, s, x);
    return __builtin_fmaf(e, 0.5f * y, s);
}

// The transforms' tables, by default the constant arrays; a kernel may pass copies in LDS.
// A gather of 64 lanes from 16-byte entries through the vector cache takes about 40 cycles
// of the CU's one address path however few lines it touches, which bounds a transform that
// makes four of them per lane; from LDS it takes about half and that path stays free.
struct math_tables
{
    const double2* nsc  = rr_nsc_tab;
    const double2* sc   = rr_bm_sctab;
    const double*  ex   = rr_exptab;
    const double*  plog = rr_plog_tab[0];
    const double*  psc  = rr_psc_tab[0];
};

// sin and cos of a Box-Muller angle v: qoff = 16 q selects q = round(128 v / pi), which the
// callers take from the word the angle came from.  The table's step is pi/128 as a double:
// with a step of 15 bits (a = v - q P exact in float) the entries next to a quarter turn
// cancel with a, and the small sine or cosine kept only 42 bits.
__host__ __device__ __forceinline__ void sincos_unit(float v, uint32_t qoff, double& s, double& c,
                                                     const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
    const double2 t  = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(tab.sc) + qoff);
    const double  a  = __builtin_fma((double)qoff, -RR_BM_ANGLE_STEP / 16, (double)v);
    const double  a2 = a * a;
    double        sa = __builtin_fma(a2, -1.0 / 5040, 1.0 / 120);
    sa               = __builtin_fma(a * a2, __builtin_fma(a2, sa, -1.0 / 6), a);
    double        ca = __builtin_fma(a2, -1.0 / 720, 1.0 / 24);
    ca               = __builtin_fma(a2, __builtin_fma(a2, ca, -0.5), 1.0);
    s                = __builtin_fma(t.x, ca, t.y * sa);
    c                = __builtin_fma(t.y, ca, -(t.x * sa));
}
__host__ __device__ __forceinline__ void sincosf_unit(float v, uint32_t qoff, float& s, float& c,
                                                      const math_tables& tab = math_tables{})
{
    double sd, cd;
    sincos_unit(v, qoff, sd, cd, tab);
    s = (float)sd;
    c = (float)cd;
}

// exp of a float, rounded to float by expf_acc: x = (32 e + j) ln2/32 + r, exp x = 2^e 2^(j/32) exp(r)
// with the 2^(j/32) table of rocrand_amd_mathtab.h.  Arguments are clamped to [-110, 100]
// first (the float result is then 0 or +inf already); a NaN passes through the clamp.
__host__ __device__ __forceinline__ double exp_acc(float xf, const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
#if defined(__HIP_DEVICE_COMPILE__)
    const float xc = __builtin_elementwise_maximum(__builtin_elementwise_minimum(xf, 100.0f), -110.0f);
#else
    const float xc = xf < -110.0f ? -110.0f : (xf > 100.0f ? 100.0f : xf);
#endif
    const float  kf = __builtin_rintf(xc * (float)RR_EXP_INV_STEP);
    const int    k  = (int)kf;
    const double kd = (double)kf;
    const double r  = __builtin_fma(kd, -RR_EXP_STEP_LO, __builtin_fma(kd, -RR_EXP_STEP_HI, (double)xc));
    double       p  = __builtin_fma(r, 1.0 / 120, 1.0 / 24);
    p               = __builtin_fma(p, r, 1.0 / 6);
    p               = __builtin_fma(p, r, 0.5);
    p               = __builtin_fma(p, r, 1.0);
    const double t  = tab.ex[k & ((1 << RR_EXPTAB_BITS) - 1)];
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ldexp(__builtin_fma(t * r, p, t), k >> RR_EXPTAB_BITS);
#else
    return __builtin_ldexp(__builtin_fma(t * r, p, t), k >> RR_EXPTAB_BITS);
#endif
}
__host__ __device__ __forceinline__ float expf_acc(float xf, const math_tables& tab = math_tables{})
{
    return (float)exp_acc(xf, tab);
}

// ---------------------------------------------------------------- double functions
// The double transforms' log, exp, sin and cos, evaluated in double-double arithmetic
// (Dekker's exact sum and product) and rounded once: each result is within
// 2^-66 (relative) of the exact value before that rounding, so it is the correctly rounded
// double except for arguments within that distance of a rounding boundary.  The
// reference's host path takes these steps through the host libm, which rounds them
// correctly but for rare hard cases; evaluated this way the device reproduces its
// intermediate values.  Host and device compile the same code (the host twin of the
// tests checks them against quad precision).
__host__ __device__ __forceinline__ void rr_two_sum(double a, double b, double& s, double& e)
{
    ROCRAND_AMD_FP_EXACT
    s               = a + b;
    const double bb = s - a;
    e               = (a - (s - bb)) + (b - bb);
}
// |a| >= |b| (or a = 0)
__host__ __device__ __forceinline__ void rr_fast_two_sum(double a, double b, double& s, double& e)
{
    ROCRAND_AMD_FP_EXACT
    s = a + b;
    e = b - (s - a);
}
__host__ __device__ __forceinline__ void rr_two_prod(double a, double b, double& p, double& e)
{
    ROCRAND_AMD_FP_EXACT
    p = a * b;
    e = __builtin_fma(a, b, -p);
}
__host__ __device__ __forceinline__ double rr_bits_to_double(uint64_t b)
{
    double x;
    __builtin_memcpy(&x, &b, sizeof(x));
    return x;
}
__host__ __device__ __forceinline__ uint64_t rr_double_to_bits(double x)
{
    uint64_t b;
    __builtin_memcpy(&b, &x, sizeof(b));
    return b;
}

// ln x: x = 2^k m, m in [sqrt(1/2), sqrt(2)), c the centre of m's table interval
// (rocrand_amd_mathtab.h), r = m/c - 1 exact as a double-double (|r| < 2^-8), and
// ln x = k ln 2 - ln(1/c) + log1p(r) with log1p to r^10.
__host__ __device__ __forceinline__ double log_cr(double x)
{
    ROCRAND_AMD_FP_EXACT
    if(!(x > 0.0) || x == __builtin_inf())
        return x == 0.0 ? -__builtin_inf() : (x > 0.0 ? x : __builtin_nan(""));
    int kadj = 0;
    if(x < 0x1p-1022)
    {
        x *= 0x1p54; // subnormal: scale into the normal range
        kadj = -54;
    }
    const uint64_t ix  = rr_double_to_bits(x);
    const uint32_t tmp = (uint32_t)(ix >> 32) - RR_DLOG_OFF;
    const int      ke  = (int)tmp >> 20;
    const double   k   = (double)(ke + kadj);
    const double   m   = rr_bits_to_double(ix - ((uint64_t)(int64_t)ke << 52));
    const double*  e   = rr_dlog_tab[(tmp >> 13) & 127u];
    double         p, pe, rh, rl;
    rr_two_prod(m, e[0], p, pe);
    rr_two_sum(p - 1.0, pe, rh, rl); // p - 1 is exact: p is within 2^-7 of 1
    const double r2  = rh * rh;
    const double r2e = __builtin_fma(rh, rh, -r2);
    double       q   = __builtin_fma(rh, -1.0 / 10, 1.0 / 9);
    q                = __builtin_fma(q, rh, -1.0 / 8);
    q                = __builtin_fma(q, rh, 1.0 / 7);
    q                = __builtin_fma(q, rh, -1.0 / 6);
    q                = __builtin_fma(q, rh, 1.0 / 5);
    q                = __builtin_fma(q, rh, -1.0 / 4);
    q                = __builtin_fma(q, rh, 1.0 / 3);
    // log1p(r) = r - r^2/2 + r^3 q(r); the tail's share of r^2 / 2 and r^3 / 3 folded below
    double a, ae, b, be, c, ce;
    rr_two_sum(k * RR_DLN2_HI, e[1], a, ae);
    rr_two_sum(a, rh, b, be);
    rr_two_sum(b, -0.5 * r2, c, ce);
    const double tail = (rl - 0.5 * r2e - rh * rl) + r2 * (rh * q + rl);
    const double lo   = (ae + be + ce) + (k * RR_DLN2_MI + e[2]) + tail;
    return c + lo;
}

// e^x: x = (64 k + j) ln2/64 + r (|r| <= ln2/128, the product with the head of ln2/64
// exact), e^x = 2^k 2^(j/64) (1 + expm1(r)) with 2^(j/64) a double-double and expm1 to r^8.
__host__ __device__ __forceinline__ double exp_cr(double x)
{
    ROCRAND_AMD_FP_EXACT
    if(x != x)
        return x;
    if(x > 709.782712893384)
        return __builtin_inf();
    if(x < -745.1332191019412)
        return 0.0;
    const double qd = __builtin_rint(x * RR_DEXP_INV_STEP);
    const int    q  = (int)qd;
    double       rh, rl;
    rr_two_sum(__builtin_fma(-qd, RR_DEXP_STEP_HI, x), -qd * RR_DEXP_STEP_MI, rh, rl);
    rl               = __builtin_fma(-qd, RR_DEXP_STEP_LO, rl);
    const double r2  = rh * rh;
    const double r2e = __builtin_fma(rh, rh, -r2);
    double       pp  = __builtin_fma(rh, 1.0 / 40320, 1.0 / 5040);
    pp               = __builtin_fma(pp, rh, 1.0 / 720);
    pp               = __builtin_fma(pp, rh, 1.0 / 120);
    pp               = __builtin_fma(pp, rh, 1.0 / 24);
    pp               = __builtin_fma(pp, rh, 1.0 / 6);
    // expm1(r) = eh + el
    const double  eh = rh;
    const double  el = __builtin_fma(0.5, r2, (rl + (0.5 * r2e + rh * rl)) + r2 * rh * pp);
    const double2 t  = rr_dexp_tab[q & 63];
    double        s1, s1e, s, se;
    rr_two_prod(t.x, eh, s1, s1e);
    rr_fast_two_sum(t.x, s1, s, se);
    const double lo = (se + s1e) + (t.x * el + t.y) + t.y * (eh + el);
    return ldexp(s + lo, q >> 6);
}

// sin t and cos t for t in [0, 2 pi + 2^-48]: t = q pi/64 + r (|r| <= pi/128, the products
// with the two heads of pi/64 exact), then the angle-addition formulas with sin(q pi/64),
// cos(q pi/64) as double-doubles and sin r to r^9, cos r to r^10.  Where sin t (cos t) is
// near 0 the table entry is an exact 0 and the result keeps its relative accuracy.
__host__ __device__ __forceinline__ void sincos_cr(double t, double& sn, double& cs)
{
    ROCRAND_AMD_FP_EXACT
    const double qd = __builtin_rint(t * RR_DSC_INV_STEP);
    const int    q  = (int)qd;
    double       rh, rl;
    rr_two_sum(__builtin_fma(-qd, RR_DSC_STEP_HI, t), -qd * RR_DSC_STEP_MI, rh, rl);
    rl               = __builtin_fma(-qd, RR_DSC_STEP_LO, rl);
    const double r2  = rh * rh;
    const double r2e = __builtin_fma(rh, rh, -r2);
    double       ps  = __builtin_fma(r2, 1.0 / 362880, -1.0 / 5040);
    ps               = __builtin_fma(ps, r2, 1.0 / 120);
    ps               = __builtin_fma(ps, r2, -1.0 / 6);
    double pc        = __builtin_fma(r2, -1.0 / 3628800, 1.0 / 40320);
    pc               = __builtin_fma(pc, r2, -1.0 / 720);
    pc               = __builtin_fma(pc, r2, 1.0 / 24);
    // sin r = rh + sl, cos r = 1 + ch + cl
    const double  sl = __builtin_fma(r2 * rh, ps, __builtin_fma(-0.5 * r2, rl, rl));
    const double  ch = -0.5 * r2;
    const double  cl = __builtin_fma(r2 * r2, pc, -(0.5 * r2e + rh * rl));
    const double* T  = rr_dsc_tab[q];
    const double  S = T[0], Sl = T[1], C = T[2], Cl = T[3];
    double        p1, p1e, p2, p2e, a, ae, b, be;
    // sin t = S cos r + C sin r
    rr_two_prod(C, rh, p1, p1e);
    rr_two_prod(S, ch, p2, p2e);
    rr_two_sum(S, p1, a, ae);
    rr_two_sum(a, p2, b, be);
    sn = b + (((ae + be) + (p1e + p2e)) + ((S * cl + C * sl) + (Sl * (1.0 + ch) + Cl * (rh + sl))));
    // cos t = C cos r - S sin r
    rr_two_prod(-S, rh, p1, p1e);
    rr_two_prod(C, ch, p2, p2e);
    rr_two_sum(C, p1, a, ae);
    rr_two_sum(a, p2, b, be);
    cs = b + (((ae + be) + (p1e + p2e)) + ((C * cl - S * sl) + (Cl * (1.0 + ch) - Sl * (rh + sl))));
}

// rocrand_uniform.h:63-66: 2^-32 + v * 2^-32.  The product by a power of two is
// exact, so one fused multiply-add rounds exactly like the separate operations.
__device__ __forceinline__ float uniform_f32(uint32_t v)
{
    return __builtin_fmaf((float)v, R_2POW32_INV, R_2POW32_INV);
}
// rocrand_uniform.h:70-73
__device__ __forceinline__ float uniform_f32(uint64_t v)
{
    return __builtin_fmaf((float)(v >> 32), R_2POW32_INV, R_2POW32_INV);
}
// rocrand_uniform.h:100-107 (53-bit integer: exact in double, exact product)
__device__ __forceinline__ double uniform_f64(uint32_t v1, uint32_t v2)
{
    const uint64_t v = (uint64_t)v1 | ((uint64_t)(v2 >> 11) << 32);
    return __builtin_fma((double)v, R_2POW53_INV_DBL, R_2POW53_INV_DBL);
}
// rocrand_uniform.h:109-116
__device__ __forceinline__ double uniform_f64(uint64_t v)
{
    return __builtin_fma((double)(v >> 11), R_2POW53_INV_DBL, R_2POW53_INV_DBL);
}
// rocrand_uniform.h:154-157
__device__ __forceinline__ __half uniform_f16(uint32_t v16)
{
    return __float2half(__builtin_fmaf((float)(v16 & 0xffffu), R_2POW16_INV, R_2POW16_INV));
}

template<int MRG>
struct mrg_consts;
template<>
struct mrg_consts<32>
{
    static constexpr double norm      = MRG32_NORM_DOUBLE;
    static constexpr double uint_norm = MRG32_UINT_NORM;
};
template<>
struct mrg_consts<31>
{
    static constexpr double norm      = MRG31_NORM_DOUBLE;
    static constexpr double uint_norm = MRG31_UINT_NORM;
};

// (double)v * k, correctly rounded, in one fused multiply-add and no integer-to-double
// conversion: the double with high word 0x43300000 and low word v is 2^52 + v exactly,
// and fma(2^52 + v, k, -2^52 k) rounds (2^52 + v) k - 2^52 k = v k once (2^52 k is exact,
// a power-of-two scaling of k).
__host__ __device__ __forceinline__ double scale_u32(uint32_t v, double k)
{
    const double x = rr_bits_to_double(0x4330000000000000ull | v);
    return __builtin_fma(x, k, -0x1p52 * k);
}

// rocrand_uniform.h:161-219
template<int MRG>
__device__ __forceinline__ uint32_t mrg_uint(uint32_t v)
{
    return (uint32_t)scale_u32(v - 1, mrg_consts<MRG>::uint_norm);
}
template<int MRG>
__host__ __device__ __forceinline__ float mrg_f32(uint32_t v)
{
    return (float)scale_u32(v, mrg_consts<MRG>::norm);
}
template<int MRG>
__device__ __forceinline__ double mrg_f64(uint32_t v)
{
    return scale_u32(v, mrg_consts<MRG>::norm);
}

// The Box-Muller pair sin(v) sqrt(-2 ln u), cos(v) sqrt(-2 ln u) for a float u in
// [2^-32, 1] and a float angle v in (0, 2 pi], evaluated in double and rounded to float
// once.  qoff = 16 q selects the angle table entry for q = round(256 v / pi), which the
// callers take from the word the angle came from (integer operations).
//   x = -2 ln u: neg2log<4>;
//   angle: v = q P + a with P = pi/256 to 15 bits, a = v - q P exact in float (|a| < 0.0063),
//     and sin v = cos a (S + C tan a), cos v = cos a (C - S tan a) with S, C = sin, cos of
//     q P from rr_nsc_tab (halved) and tan a = a + g a^3 (g the best for that range, a little
//     over 1/3: relative error 2^-34);
//   radius times cos a: with y the hardware's reciprocal square root of x and t = x y, one
//     Newton step gives 2 sqrt(x) = t (3 - t y) to 2^-46, and as 3 - t y is 2 to 2^-23,
//     2 sqrt(x) cos a = t (3 - a^2 - t y) to 2^-33: the cosine costs no product of its own.
//     The doubling is the table's half; the radius keeps the sign of a zero.
// The pair before its rounding is within 2^-31 of exact, so each output is within 0.508
// ulp of the exact value, and within 2 ulp of the reference's float pipeline (logf, sqrtf,
// sinf/cosf and the product: four roundings, rocrand_normal.h:51-66).  About 34 VALU
// operations a pair (38 with sin and cos as sums of products with sin a and cos a and a
// separate radius; XORWOW normal f32, 2^27 values, with its table in LDS: 3.30 -> 3.87
// TB/s).  UNIT rounds
// sin(v) s + 0 instead of sin(v) s: the output of mean + 1 * x at mean +0 (a zero is +0).
template<bool UNIT = false>
__host__ __device__ __forceinline__ void box_muller_dd(float u, float v, uint32_t qoff, float& r0, float& r1,
                                                       const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
    const double  x  = neg2log<4>(u);
    const double2 st = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(tab.nsc) + qoff);
    const double  a  = (double)__builtin_fmaf(-(float)qoff, RR_NSC_STEP * 0.0625f, v);
    const double  c3 = __builtin_fma(-a, a, 3.0);
    constexpr double g = 1.0 / 3 + 4.3e-6;
    const double  ta = a * __builtin_fma(c3, -g, 1.0 + 3.0 * g); // a (1 + g a^2)
    const double  y  = rr_rsq(__builtin_fmax(x, 0x1p-126));
    const double  t  = x * y;
    const double  s  = t * __builtin_fma(-t, y, c3);
    const double  sn = __builtin_fma(st.y, ta, st.x);
    const double  cs = __builtin_fma(-st.x, ta, st.y);
    if constexpr(UNIT)
    {
        r0 = (float)__builtin_fma(sn, s, 0.0);
        r1 = (float)__builtin_fma(cs, s, 0.0);
    }
    else
    {
        r0 = (float)(sn * s);
        r1 = (float)(cs * s);
    }
}

// rocrand_normal.h:51-66: u = 2^-32 + x 2^-32, angle 2^-32 2pi + y 2^-32 2pi (rounded as
// the reference rounds them), then the pair above; the angle is about 2 pi (y + 1) 2^-32,
// so q = round(y 2^-23) (and for the 257-entry table of the stepwise pair, round(y 2^-24)).
template<bool UNIT = false>
__device__ __forceinline__ void box_muller(uint32_t x, uint32_t y, float& r0, float& r1,
                                           const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
    const float u = uniform_f32(x);
    const float v = R_2POW32_INV_2PI + (float)y * R_2POW32_INV_2PI;
    box_muller_dd<UNIT>(u, v, ((y >> 19) + 8u) & ~15u, r0, r1, tab);
}

// The same pair through the reference's own steps -- logf, sqrtf, sinf/cosf, each rounded
// to float (correctly) -- for the log-normal transforms: exp magnifies a one-ulp change
// of the variate to several ulps of the output, and these steps reproduce the reference
// host path's variate bit for bit wherever its libm rounds correctly.
__device__ __forceinline__ void box_muller_uv_stepwise(float u, float v, uint32_t qoff, float& r0, float& r1,
                                                       const math_tables& tab)
{
    ROCRAND_AMD_FP_EXACT
    const float s = sqrtf_unit((float)neg2log<6>(u));
    float       sn, cs;
    sincosf_unit(v, qoff, sn, cs, tab);
    r0 = sn * s;
    r1 = cs * s;
}
__device__ __forceinline__ void box_muller_stepwise(uint32_t x, uint32_t y, float& r0, float& r1,
                                                    const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
    const float u = uniform_f32(x);
    const float v = R_2POW32_INV_2PI + (float)y * R_2POW32_INV_2PI;
    box_muller_uv_stepwise(u, v, ((y >> 20) + 8u) & ~15u, r0, r1, tab);
}
// rocrand_normal.h:76-96 (host branch: sin(w * pi), not sincospi).
__device__ __forceinline__ void box_muller_double(uint32_t a, uint32_t b, uint32_t c, uint32_t d, double& r0,
                                                  double& r1)
{
    ROCRAND_AMD_FP_EXACT
    const uint64_t v1 = (uint64_t)a ^ ((uint64_t)b << 21);
    const double   u  = R_2POW53_INV_DBL + (double)v1 * R_2POW53_INV_DBL;
    const uint64_t v2 = (uint64_t)c ^ ((uint64_t)d << 21);
    const double   w  = R_2POW53_INV_DBL * 2.0 + (double)v2 * (R_2POW53_INV_DBL * 2.0);
    const double   s  = __builtin_sqrt(-2.0 * log_cr(u));
    const double   t  = w * R_PI_DBL;
    double         sn, cs;
    sincos_cr(t, sn, cs);
    r0 = sn * s;
    r1 = cs * s;
}
// The double Box-Muller pair evaluated as double-doubles and rounded once, for a double u
// in [2^-53, 1] and a double angle t in (0, 2 pi + 2^-48]; qoff = 32 q selects the angle
// table entry for q = round(128 t / pi), which the callers take from the angle's word.
//   x = -2 ln u: u = 2^k m, a = a multiple of 2^-8 next to 1/m (rr_plog_tab), so r = m a - 1
//     is exact (|r| < 2^-7.3), and x = (-2 k ln 2 + 2 ln a) - 2 r + r^2 (1 - 2/3 r + ...):
//     the first two terms add exactly in their heads, the sums with 2 r and with the rest
//     (to r^8, small enough to be a double) leave their rounding errors in the tail;
//   sqrt: t1 = sqrt(x) to 2^-46 from the hardware's reciprocal square root and a step, and
//     the exact residual x - t1^2 gives the tail;
//   angle: a = t - q P is exact for P = pi/128 rounded to double; sin and cos of q P as
//     double-doubles, the products with a and the sums carried with their errors.
// Relative error below 2^-58 before the rounding: within 0.52 ulp of the exact value, where
// the reference's steps (log, sqrt, sin/cos and product, rounded one by one) may be 2.3
// ulp off, and within 2 ulp of those.  Next to a quarter turn (an MRG's float angle is
// exactly one for one pair in some 10^7) the small sine or cosine is the table entry's tail,
// itself a rounded double, so that value is within 1 ulp (0.89 the largest of 2.6e7 there),
// and the head's part of the radius' tail alone would leave it 40 ulp off: hence
// (sn + se) tl and (cs + ce) tl.  117 VALU instructions with its uniforms and the affine
// step; taking those steps one by one, each correctly rounded, costs 243 (2^28 normal f64
// values: XORWOW 2.08 -> 3.51 TB/s, MRG32k3a 2.06 -> 3.51, Philox 2.01 -> 3.09).
__host__ __device__ __forceinline__ void box_muller_pair_double(double u, double t, uint32_t qoff, double& r0,
                                                                double& r1, const math_tables& tab)
{
    ROCRAND_AMD_FP_EXACT
    // x = xh + xl
    const uint64_t ix  = rr_double_to_bits(u);
    const uint32_t hw  = (uint32_t)(ix >> 32), tmp = hw - RR_DLOG_OFF;
    const double   k   = (double)((int32_t)tmp >> 20);
    const double   m   = rr_bits_to_double(((uint64_t)(hw - (tmp & 0xfff00000u)) << 32) | (uint32_t)ix);
    const double*  lt  = reinterpret_cast<const double*>(reinterpret_cast<const char*>(tab.plog)
                                                       + ((tmp >> 8) & 0xfe0u));
    const double   r   = __builtin_fma(m, lt[0], -1.0);
    double         p   = __builtin_fma(r, 1.0 / 4, -2.0 / 7);
    p                  = __builtin_fma(p, r, 1.0 / 3);
    p                  = __builtin_fma(p, r, -2.0 / 5);
    p                  = __builtin_fma(p, r, 1.0 / 2);
    p                  = __builtin_fma(p, r, -2.0 / 3);
    p                  = __builtin_fma(p, r, 1.0);
    const double s0    = __builtin_fma(k, RR_PLOG_M2LN2_HI, lt[1]);
    const double sl    = __builtin_fma(k, RR_PLOG_M2LN2_LO, lt[2]);
    const double x1    = __builtin_fma(-2.0, r, s0);
    const double q     = __builtin_fma(r * r, p, sl);
    const double xh    = x1 + q;
    const double xl    = __builtin_fma(-2.0, r, -(x1 - s0)) + (q - (xh - x1));
    // sqrt(x) = th + tl
    const double y     = rr_rsq(__builtin_fmax(xh, 0x1p-126));
    const double h     = 0.5 * y;
    const double g     = xh * y;
    const double th    = __builtin_fma(__builtin_fma(-g, g, xh), h, g);
    const double tl    = (__builtin_fma(-th, th, xh) + xl) * h;
    // a = t - q P; sin a = a + sa, cos a = 1 + ca
    const double* T    = reinterpret_cast<const double*>(reinterpret_cast<const char*>(tab.psc) + qoff);
    const double  S = T[0], Sl = T[1], C = T[2], Cl = T[3];
    const double  a    = __builtin_fma((double)qoff, -RR_PSC_STEP / 32, t);
    const double  a2   = a * a;
    const double  sa   = a * a2 * __builtin_fma(a2, __builtin_fma(a2, -1.0 / 5040, 1.0 / 120), -1.0 / 6);
    const double  ca   = a2 * __builtin_fma(a2, __builtin_fma(a2, -1.0 / 720, 1.0 / 24), -0.5);
    // sin t = S cos a + C sin a = sn + se
    const double  p1   = C * a;
    const double  sn   = S + p1;
    double        se   = p1 - (sn - S);
    se                 = __builtin_fma(S, ca, se);
    se                 = __builtin_fma(C, sa, se);
    se                 = __builtin_fma(Cl, a, se + __builtin_fma(C, a, -p1) + Sl);
    // cos t = C cos a - S sin a = cs + ce
    const double  p2   = S * a;
    const double  cs   = C - p2;
    double        ce   = (C - cs) - p2;
    ce                 = __builtin_fma(C, ca, ce);
    ce                 = __builtin_fma(-S, sa, ce);
    ce                 = __builtin_fma(-Sl, a, ce - __builtin_fma(S, a, -p2) + Cl);
    // the products, rounded once
    const double  q0   = sn * th, q1 = cs * th;
    r0 = q0 + __builtin_fma(se, th, __builtin_fma(sn + se, tl, __builtin_fma(sn, th, -q0)));
    r1 = q1 + __builtin_fma(ce, th, __builtin_fma(cs + ce, tl, __builtin_fma(cs, th, -q1)));
}
// The pair of four words: u = (v1 + 1) 2^-53 and w = (v2 + 1) 2^-52 rounded to double, each
// from its word's halves in two exact fused operations and one rounding (rocrand_normal.h:76-96);
// the angle is about 2 pi v2 2^-53, and v2's high word is d >> 11.
__host__ __device__ __forceinline__ void normal_pair_double(uint32_t a, uint32_t b, uint32_t c, uint32_t d, double& r0,
                                                            double& r1, const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
    const double u = __builtin_fma((double)(b >> 11), 0x1p-21,
                                   __builtin_fma((double)(a ^ (b << 21)), R_2POW53_INV_DBL, R_2POW53_INV_DBL));
    const double w = __builtin_fma((double)(d >> 11), 0x1p-20,
                                   __builtin_fma((double)(c ^ (d << 21)), 0x1p-52, 0x1p-52));
    box_muller_pair_double(u, w * R_PI_DBL, (((d >> 11) + 4096u) >> 8) & ~31u, r0, r1, tab);
}
// rocrand_normal.h:108-135, host (float math) branch.
__device__ __forceinline__ void box_muller_half(uint32_t x16, uint32_t y16, float& h0, float& h1,
                                                const math_tables& tab)
{
    ROCRAND_AMD_FP_EXACT
    const float u = R_2POW16_INV + (float)(x16 & 0xffffu) * R_2POW16_INV;
    const float v = R_2POW16_INV_2PI + (float)(y16 & 0xffffu) * R_2POW16_INV_2PI;
    float       r0, r1; // the angle is about 2 pi (y16 + 1) 2^-16
    box_muller_uv_stepwise(u, v, (((y16 & 0xffffu) >> 4) + 8u) & ~15u, r0, r1, tab);
    h0 = __half2float(__float2half(r0));
    h1 = __half2float(__float2half(r1));
}
// rocrand_normal.h:138-154
// The MRG outputs y in [1, m] scale by about 2^-32 (MRG32k3a) or 2^-31 (MRG31k3p), so
// q = round(y 2^-23) or round(y 2^-22) (stepwise pair: round(y 2^-24) or round(y 2^-23)).
template<int MRG, bool UNIT = false>
__device__ __forceinline__ void mrg_box_muller(uint32_t x, uint32_t y, float& r0, float& r1,
                                               const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
    constexpr int SH = MRG == 32 ? 19 : 18;
    box_muller_dd<UNIT>(mrg_f32<MRG>(x), mrg_f32<MRG>(y) * R_2PI, ((y >> SH) + 8u) & ~15u, r0, r1, tab);
}
template<int MRG>
__device__ __forceinline__ void mrg_box_muller_stepwise(uint32_t x, uint32_t y, float& r0, float& r1,
                                                        const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
    constexpr int SH = MRG == 32 ? 20 : 19;
    box_muller_uv_stepwise(mrg_f32<MRG>(x), mrg_f32<MRG>(y) * R_2PI, ((y >> SH) + 8u) & ~15u, r0, r1, tab);
}
// rocrand_normal.h:156-172: float-precision uniforms widened to double.
template<int MRG>
__device__ __forceinline__ void mrg_box_muller_double(uint32_t x, uint32_t y, double& r0, double& r1)
{
    ROCRAND_AMD_FP_EXACT
    const double u = (double)mrg_f32<MRG>(x);
    const double v = (double)mrg_f32<MRG>(y) * 2.0;
    const double s = __builtin_sqrt(-2.0 * log_cr(u));
    double       sn, cs;
    sincos_cr(v * R_PI_DBL, sn, cs);
    r0 = sn * s;
    r1 = cs * s;
}
// The pair of rocrand_normal.h:156-172 evaluated as double-doubles and rounded once.
template<int MRG>
__host__ __device__ __forceinline__ void mrg_normal_pair_double(uint32_t x, uint32_t y, double& r0, double& r1,
                                                                const math_tables& tab = math_tables{})
{
    ROCRAND_AMD_FP_EXACT
    constexpr int SH = MRG == 32 ? 19 : 18;
    const double  v  = (double)mrg_f32<MRG>(y) * 2.0;
    box_muller_pair_double((double)mrg_f32<MRG>(x), v * R_PI_DBL, ((y >> SH) + 16u) & ~31u, r0, r1, tab);
}
// rocrand_normal.h:199-221 roc_d_erfinv and :263-268 normal_distribution_double.
__device__ __forceinline__ double roc_d_erfinv(double x)
{
    ROCRAND_AMD_FP_EXACT
    const double sgn = (x < 0.0) ? -1.0 : 1.0;
    x                = (1.0 - x) * (1.0 + x);
    const double lnx = log_cr(x);
    if(isnan(lnx))
        return 1.0;
    if(isinf(lnx))
        return 0.0;
    const double tt1 = 2.0 / (R_PI_DBL * 0.147) + 0.5 * lnx;
    const double tt2 = 1.0 / 0.147 * lnx;
    return sgn * __builtin_sqrt(-tt1 + __builtin_sqrt(tt1 * tt1 - tt2));
}
__device__ __forceinline__ double normal_double_1(double p)
{
    ROCRAND_AMD_FP_EXACT
    return (double)R_SQRT2 * roc_d_erfinv(2.0 * p - 1.0);
}

// rocrand_normal.h:174-197 roc_f_erfinv, float arithmetic rounded step by step.  x is 0 or
// the difference of two floats of [0, 1], so (1 - x)(1 + x) is 0 or in [2^-23, 1]; at 0
// (the logarithm is -inf) the reference returns 0.  The roots' arguments are 0 or at least
// ulp(4.33).
__device__ __forceinline__ float roc_f_erfinv(float x)
{
    ROCRAND_AMD_FP_EXACT
    const float     z   = (1.0f - x) * (1.0f + x);
    const float     lnx = logf_unit(z > 0.0f ? z : 1.0f);
    constexpr float c1  = 2.0f / (3.141592653f * 0.147f);
    constexpr float c2  = 1.0f / 0.147f;
    const float     tt1 = c1 + 0.5f * lnx;
    const float     tt2 = c2 * lnx;
    const float     w   = sqrtf_unit(-tt1 + sqrtf_unit(tt1 * tt1 - tt2));
    return z > 0.0f ? __builtin_copysignf(w, x) : 0.0f;
}

// Uniforms of a direction value (rocrand_uniform.h:63-116 on the 32- or 64-bit value).
__device__ __forceinline__ float sob_uf32(uint32_t x) { return uniform_f32(x); }
__device__ __forceinline__ float sob_uf32(uint64_t x) { return uniform_f32(x); }
__device__ __forceinline__ double sob_uf64(uint32_t x)
{
    return __builtin_fma((double)x, R_2POW32_INV_DBL, R_2POW32_INV_DBL);
}
__device__ __forceinline__ double sob_uf64(uint64_t x) { return uniform_f64(x); }

// rocrand_normal.h:228-296 normal_distribution(_double) on a direction value.
template<class V>
__device__ __forceinline__ float sob_normal_f32(V x)
{
    ROCRAND_AMD_FP_EXACT
    const float p = sob_uf32(x);
    return R_SQRT2 * roc_f_erfinv(2.0f * p - 1.0f);
}
template<class V>
__device__ __forceinline__ double sob_normal_f64(V x)
{
    return normal_double_1(sob_uf64(x));
}

} // namespace rocrand_amd_engine

