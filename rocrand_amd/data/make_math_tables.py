"""Write include/rocrand/rocrand_amd_mathtab.h: the tables of the float-argument logarithm
(Box-Muller radius), sine and cosine (Box-Muller angle) and exponential (log-normal
outputs) evaluated in double, and of the double transforms.

Exponential, 32 entries: 2^(j/32) rounded to double, j = 0..31; with x = (32 e + j) ln2/32
+ r, |r| <= ln2/64, exp x = 2^e 2^(j/32) exp(r).  The reduction constant ln2/32 is split
into a head with its low 16 bits clear (exact products with |32 e + j| < 2^16) and the
rounded remainder.

Box-Muller pair (evaluated in double and rounded once), logarithm, 33 x 64 entries: a
float u in [2^-32, 1] with bit pattern b has biased exponent e = b >> 23 in [95, 127] and
interval i = bits 17..22 of b (z = u 2^(127-e) in [1 + i/64, 1 + (i+1)/64)).  Entry
(e - 95) * 64 + i holds a = 2^(127-e) / c, c the centre of the interval, and
b = -2 ln(u / (a u)) = -2 ((e - 127) ln 2 + ln c) for the rounded a, so that
-2 ln u = b - 2 log1p(u a - 1), |u a - 1| < 2^-7.  The interval [1, 1 + 1/64) of e = 127
holds only u = 1: its entry is a = 1, b = -0, which gives -2 ln 1 = -0 (the reference's
-2.0f * logf(1.0f)).  The last interval below 1, u in [1 - 2^-7, 1), takes c = 1 (a = 1,
b = 0) instead of its centre: r = u - 1 is then exact and small with ln u, so -2 ln u
keeps its relative accuracy where it approaches 0.

Box-Muller sine and cosine, 257 entries: angles q P, q = 0..256, P = pi/128 rounded to
double (v - q P rounds once, |v - q P| < 0.0124); entry q holds sin(q P), cos(q P) rounded to
double, which at a quarter turn is at most 2.5e-16, so that the small sine or cosine next to
one is v - q P itself and nothing cancels.

Float normals, sine and cosine, 513 entries: angles q P, q = 0..512, P = pi/256 rounded to 15
significant bits (q P and v - q P are exact in float for the angles v the transform sees, |v - q P| < 0.0063); entry q holds
sin(q P)/2, cos(q P)/2 rounded to double (the radius comes out doubled).

Double-precision Box-Muller pair (evaluated as double-doubles and rounded once):
  log, 128 entries: x = 2^k m split as below; entry i holds a = a multiple of 2^-8 next to
    1/c (exactly 1 for the interval that contains 1), so that m a - 1 is exact in double,
    and 2 ln a as a head that is a multiple of 2^-42 (-0 where a = 1) and a tail; -2 ln 2 is
    split the same way, so k (-2 ln 2) + 2 ln a adds exactly in the heads.
  sin/cos, 257 entries: sin(q P) and cos(q P), q = 0..256, P = pi/128 rounded to double
    (t - q P, |t - q P| < 2^-6, is a multiple of 2^-58 or of t's last bit where that is
    smaller, so exact in double), as double-doubles; an entry next to a zero of the function
    (q P is within 2^-51 of it) is all tail.

Double-precision logarithm, exponential and sine/cosine (the double log-normals' steps,
each evaluated in double-double and rounded once):
  log, 128 entries: x = 2^k m with the high word of m in [0x3fe6a09e, 0x3ff6a09e)
    (m in [sqrt(1/2), sqrt(2))); entry i covers the m whose high word minus 0x3fe6a09e has
    bits 13..19 equal to i and holds inv = 1/c for the centre c of that interval (rounded
    to double; exactly 1 for the interval that contains 1) and -ln(inv) as a double-double.
    Then ln x = k ln 2 - ln(inv) + log1p(m inv - 1), |m inv - 1| < 2^-8.
  exp, 64 entries: 2^(j/64) as a double-double; x = (64 k + j) ln2/64 + r, |r| <= ln2/128.
  sin/cos, 129 entries: sin(q pi/64) and cos(q pi/64), q = 0..128, as double-doubles (exact
    0 and +-1 at multiples of pi/2); t = q pi/64 + r, |r| <= pi/128.
The reduction constants ln 2, ln 2/64 and pi/64 are split into heads with enough low bits
clear that their products with the integer multiples the arguments need are exact.

    python rocrand_amd/data/make_math_tables.py
"""
import os
import struct

import mpmath

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(os.path.dirname(os.path.dirname(HERE)), "include", "rocrand", "rocrand_amd_mathtab.h")
N_EXP = 32


def exp_entries():
    return [float(mpmath.power(2, mpmath.mpf(j) / N_EXP)) for j in range(N_EXP)]


BM_EMIN = 95  # biased exponent of 2^-32
BM_EMAX = 127


def bm_log_entries():
    out = []
    for e in range(BM_EMIN, BM_EMAX + 1):
        scale = mpmath.power(2, BM_EMAX - e)
        for i in range(64):
            if e == BM_EMAX and i == 0:
                out.append((1.0, -0.0))
                continue
            if e == BM_EMAX - 1 and i == 63:
                # u in [1 - 2^-7, 1): c = 1, so r = u - 1 exactly and -2 ln u keeps its
                # relative accuracy as u approaches 1
                out.append((1.0, 0.0))
                continue
            lo = 1 + mpmath.mpf(i) / 64
            c = lo + mpmath.mpf(1) / 128
            a = float(scale / c)
            # -2 ln u = -2 ln(u a) + 2 ln a, exactly, for the rounded a
            b = float(2 * mpmath.log(mpmath.mpf(a)))
            out.append((a, b))
    return out


def bm_sincos_entries():
    p = mpmath.mpf(float(mpmath.pi / 128))
    return [(float(mpmath.sin(q * p)), float(mpmath.cos(q * p))) for q in range(257)]


def rounded_to(x, bits):
    m, e = mpmath.frexp(x)
    return mpmath.nint(m * 2**bits) * mpmath.power(2, e - bits)


def normal_sincos_entries():
    p = rounded_to(mpmath.pi / 256, 15)
    return [(float(mpmath.sin(q * p) / 2), float(mpmath.cos(q * p) / 2)) for q in range(513)]


def pair_log_split(x):
    head = float(mpmath.nint(x * 2**42) / 2**42)
    return head, float(x - mpmath.mpf(head))


def pair_log_entries():
    out = []
    for i in range(128):
        lo = mpmath.mpf(f64_from_high(DLOG_OFF + i * 0x2000))
        hi = mpmath.mpf(f64_from_high(DLOG_OFF + (i + 1) * 0x2000))
        if lo <= 1 < hi:
            out.append((1.0, -0.0, 0.0))
            continue
        a = float(mpmath.nint(2 / (lo + hi) * 256) / 256)
        out.append((a, *pair_log_split(2 * mpmath.log(mpmath.mpf(a)))))
    return out


def pair_sincos_entries():
    p = mpmath.mpf(float(mpmath.pi / 128))

    def tail_if_zero(x):
        return (0.0, float(x)) if abs(x) < mpmath.power(2, -30) else dd(x)

    return [(*tail_if_zero(mpmath.sin(q * p)), *tail_if_zero(mpmath.cos(q * p))) for q in range(257)]


DLOG_OFF = 0x3FE6A09E


def f64_from_high(hw):
    return struct.unpack("<d", struct.pack("<Q", hw << 32))[0]


def dd(x):
    hi = float(x)
    return hi, float(x - mpmath.mpf(hi))


def dlog_entries():
    out = []
    for i in range(128):
        lo = mpmath.mpf(f64_from_high(DLOG_OFF + i * 0x2000))
        hi = mpmath.mpf(f64_from_high(DLOG_OFF + (i + 1) * 0x2000))
        if lo <= 1 < hi:
            out.append((1.0, 0.0, 0.0))
            continue
        inv = float(2 / (lo + hi))
        t_hi, t_lo = dd(-mpmath.log(mpmath.mpf(inv)))
        out.append((inv, t_hi, t_lo))
    return out


def dexp_entries():
    return [dd(mpmath.power(2, mpmath.mpf(j) / 64)) for j in range(64)]


def dsincos_entries():
    out = []
    for q in range(129):
        if q % 32 == 0:
            k = q // 32
            out.append(([0.0, 1.0, 0.0, -1.0, 0.0][k], 0.0, [1.0, 0.0, -1.0, 0.0, 1.0][k], 0.0))
            continue
        a = q * mpmath.pi / 64
        s_hi, s_lo = dd(mpmath.sin(a))
        c_hi, c_lo = dd(mpmath.cos(a))
        out.append((s_hi, s_lo, c_hi, c_lo))
    return out


def split3(c, clear_bits):
    """c = h + m + l with h and m rounded to 53 - clear_bits significant bits."""
    parts = []
    rest = mpmath.mpf(c)
    for _ in range(2):
        m, e = mpmath.frexp(rest)
        keep = 53 - clear_bits
        v = mpmath.nint(m * 2**keep) * mpmath.power(2, e - keep)
        parts.append(float(v))
        rest = rest - v
    parts.append(float(rest))
    return parts


def split(c, clear_bits):
    head = float(c)
    bits = struct.unpack("<Q", struct.pack("<d", head))[0] & ~((1 << clear_bits) - 1)
    head = struct.unpack("<d", struct.pack("<Q", bits))[0]
    return head, float(c - mpmath.mpf(head))


def ln2_split():
    head, tail = split(mpmath.log(2) / N_EXP, 16)
    return head, tail, float(N_EXP / mpmath.log(2))


def main():
    mpmath.mp.prec = 200
    exp_rows = "\n".join(f"    {a.hex()}," for a in exp_entries())
    head, tail, inv = ln2_split()
    dlog_rows = "\n".join(f"    {{{a.hex()}, {b.hex()}, {c.hex()}, 0.0}}," for a, b, c in dlog_entries())
    dexp_rows = "\n".join(f"    {{{a.hex()}, {b.hex()}}}," for a, b in dexp_entries())
    dsc_rows = "\n".join(f"    {{{a.hex()}, {b.hex()}, {c.hex()}, {d.hex()}}}," for a, b, c, d in dsincos_entries())
    ln2 = split3(mpmath.log(2), 11)            # k ln2 exact for |k| < 2^11
    l64 = split3(mpmath.log(2) / 64, 17)       # q ln2/64 exact for |q| < 2^17
    p64 = split3(mpmath.pi / 64, 8)            # q pi/64 exact for q < 2^8
    bm_log_rows = "\n".join(f"    {{{a.hex()}, {b.hex()}}}," for a, b in bm_log_entries())
    bm_sc_rows = "\n".join(f"    {{{a.hex()}, {b.hex()}}}," for a, b in bm_sincos_entries())
    bm_p = float(mpmath.pi / 128)
    nsc_rows = "\n".join(f"    {{{a.hex()}, {b.hex()}}}," for a, b in normal_sincos_entries())
    nsc_p = float(rounded_to(mpmath.pi / 256, 15))
    plog_rows = "\n".join(f"    {{{a.hex()}, {b.hex()}, {c.hex()}, 0.0}}," for a, b, c in pair_log_entries())
    psc_rows = "\n".join(f"    {{{', '.join(x.hex() for x in row)}}}," for row in pair_sincos_entries())
    m2ln2 = pair_log_split(-2 * mpmath.log(2))
    psc_p = float(mpmath.pi / 128)
    text = f"""// rocrand_amd_mathtab.h -- generated by rocrand_amd/data/make_math_tables.py; do not edit.
// Tables of the double-evaluated float logarithm, sine/cosine and exponential (rocrand_amd_math.h).
#pragma once

#include <hip/hip_runtime.h>

// Device code reads the tables from constant memory; host code (the double functions are
// also host functions) from ordinary host arrays with the same values.
#if defined(__HIP_DEVICE_COMPILE__)
#define RR_MATH_TABLE static __constant__
#else
#define RR_MATH_TABLE static
#endif

namespace rocrand_amd_engine
{{
constexpr int    RR_EXPTAB_BITS  = 5;
constexpr double RR_EXP_INV_STEP = {inv.hex()}; // {N_EXP} / ln 2
constexpr double RR_EXP_STEP_HI  = {head.hex()}; // ln 2 / {N_EXP}, low 16 bits clear
constexpr double RR_EXP_STEP_LO  = {tail.hex()}; // ln 2 / {N_EXP} - RR_EXP_STEP_HI
// 2^(j/{N_EXP})
RR_MATH_TABLE const double rr_exptab[{N_EXP}] = {{
{exp_rows}
}};

// Box-Muller pair: {{2^(127-e)/c, 2 ln(2^(127-e)/c)}} for biased exponents e = {BM_EMIN}..{BM_EMAX}
constexpr uint32_t RR_BM_EMIN = {BM_EMIN}u;
RR_MATH_TABLE const double2 rr_bm_logtab[{(BM_EMAX - BM_EMIN + 1) * 64}] = {{
{bm_log_rows}
}};
constexpr double RR_BM_ANGLE_STEP = {bm_p.hex()}; // pi/128 rounded to double
// {{sin(q RR_BM_ANGLE_STEP), cos(q RR_BM_ANGLE_STEP)}}, q = 0..256
RR_MATH_TABLE const double2 rr_bm_sctab[257] = {{
{bm_sc_rows}
}};

// Float normals' angle: {{sin(q RR_NSC_STEP)/2, cos(q RR_NSC_STEP)/2}}, q = 0..512
constexpr float RR_NSC_STEP = {nsc_p.hex()}f; // pi/256 to 15 bits
RR_MATH_TABLE const double2 rr_nsc_tab[513] = {{
{nsc_rows}
}};

// Double Box-Muller pair: {{a, 2 ln a (head, tail), 0}} for m in [sqrt(1/2), sqrt(2))
RR_MATH_TABLE const double rr_plog_tab[128][4] = {{
{plog_rows}
}};
constexpr double RR_PLOG_M2LN2_HI = {m2ln2[0].hex()}; // -2 ln 2
constexpr double RR_PLOG_M2LN2_LO = {m2ln2[1].hex()};
constexpr double RR_PSC_STEP = {psc_p.hex()}; // pi/128 rounded to double
// {{sin(q RR_PSC_STEP), cos(q RR_PSC_STEP)}} (heads, tails), q = 0..256
RR_MATH_TABLE const double rr_psc_tab[257][4] = {{
{psc_rows}
}};

// Double-precision log: {{1/c, -ln(1/c) (head, tail), 0}} for m in [sqrt(1/2), sqrt(2))
constexpr uint32_t RR_DLOG_OFF = 0x{DLOG_OFF:08x}u;
RR_MATH_TABLE const double rr_dlog_tab[128][4] = {{
{dlog_rows}
}};
constexpr double RR_DLN2_HI = {ln2[0].hex()};
constexpr double RR_DLN2_MI = {ln2[1].hex()};
constexpr double RR_DLN2_LO = {ln2[2].hex()};
// Double-precision exp: 2^(j/64) (head, tail)
RR_MATH_TABLE const double2 rr_dexp_tab[64] = {{
{dexp_rows}
}};
constexpr double RR_DEXP_INV_STEP = {float(64 / mpmath.log(2)).hex()}; // 64 / ln 2
constexpr double RR_DEXP_STEP_HI  = {l64[0].hex()};
constexpr double RR_DEXP_STEP_MI  = {l64[1].hex()};
constexpr double RR_DEXP_STEP_LO  = {l64[2].hex()};
// Double-precision sin/cos: sin(q pi/64), cos(q pi/64) (heads, tails), q = 0..128
RR_MATH_TABLE const double rr_dsc_tab[129][4] = {{
{dsc_rows}
}};
constexpr double RR_DSC_INV_STEP = {float(64 / mpmath.pi).hex()}; // 64 / pi
constexpr double RR_DSC_STEP_HI  = {p64[0].hex()};
constexpr double RR_DSC_STEP_MI  = {p64[1].hex()};
constexpr double RR_DSC_STEP_LO  = {p64[2].hex()};
}} // namespace rocrand_amd_engine
"""
    with open(OUT, "w") as f:
        f.write(text)
    print(f"wrote {OUT}")


if __name__ == "__main__":
    main()
