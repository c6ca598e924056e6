/* Host twin of the normal and log-normal transforms' functions
 * (include/rocrand/rocrand_amd_math.h: logf_unit, sincosf_unit, expf_acc, box_muller_dd,
 * normal_pair_double): the same source compiled for the host, checked against long double
 * and quad precision and against the reference's steps over this libm.  The device's
 * reciprocal square roots are emulated to their precision (2^-24).
 *
 * usage: normal_twin N
 * prints NAME COUNT VALUES  for the float functions' results that are not the correctly
 * rounded ones, and  NAME VALUES MAX_ERR_MICROULP BEYOND_2ULP_OF_LIBM  for the pairs.
 */
#include <rocrand/rocrand_amd_math.h>

#if !defined(__HIP_DEVICE_COMPILE__)
#include <math.h>
#include <quadmath.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

using namespace rocrand_amd_engine;

static uint64_t g_state = 0x9E3779B97F4A7C15ull;
static uint64_t next64()
{
    g_state ^= g_state << 13;
    g_state ^= g_state >> 7;
    g_state ^= g_state << 17;
    return g_state;
}
template<class F, class I>
static long ulps(F a, F b) // representable values between a and b
{
    I x, y;
    memcpy(&x, &a, sizeof(F));
    memcpy(&y, &b, sizeof(F));
    const I low = (I)1 << (8 * sizeof(F) - 1);
    x = x < 0 ? low - x : x;
    y = y < 0 ? low - y : y;
    return labs((long)(x - y));
}
template<class F>
static double error(F got, __float128 exact)
{
    const F e  = fabs((F)exact);
    const F sp = nextafter(e, (F)INFINITY) - e;
    return (double)(fabsq((__float128)got - exact) / (__float128)sp);
}
// words at the ends of their range and next to the angle table's boundaries, then random
static uint32_t word(long i)
{
    static const uint32_t edge[] = {0u, 1u, 0x1fffffu, 0x200000u, 0x7fffffu, 0x800000u, 0x3fffffffu, 0x40000000u,
                                    0x7fffffffu, 0x80000000u, 0xbfffffffu, 0xffbfffffu, 0xffffff7fu, 0xffffff80u,
                                    0xffffffffu};
    constexpr long        n = sizeof(edge) / sizeof(edge[0]);
    return i < n ? edge[i] : (uint32_t)(next64() >> 13);
}

int main(int argc, char** argv)
{
    const long n = argc > 1 ? atol(argv[1]) : 100000;
    long       bad = 0, total = 0;
    for(uint32_t b = 0x2f800000u; b <= 0x3f800000u; b += 257, total++)
    {
        float u;
        memcpy(&u, &b, 4);
        bad += logf_unit(u) != (float)logl((long double)u);
    }
    printf("log %ld %ld\n", bad, total);
    bad = total = 0;
    for(uint64_t y = 0; y <= 0xffffffffull; y += 257, total += 2)
    {
        const float v = R_2POW32_INV_2PI + (float)(uint32_t)y * R_2POW32_INV_2PI;
        float       s, c;
        sincosf_unit(v, (((uint32_t)y >> 20) + 8u) & ~15u, s, c);
        bad += (s != (float)sinl((long double)v)) + (c != (float)cosl((long double)v));
    }
    printf("sincos %ld %ld\n", bad, total);
    bad = total = 0;
    for(uint64_t b = 0; b <= 0xffffffffull; b += 257)
    {
        const uint32_t bb = (uint32_t)b;
        float          x;
        memcpy(&x, &bb, 4);
        if(!(x > -105.0f && x < 90.0f))
            continue;
        total++;
        bad += expf_acc(x) != (float)expl((long double)x);
    }
    printf("exp %ld %ld\n", bad, total);
    double worst = 0.0;
    long   beyond = 0;
    for(long i = 0; i < n; i++)
    {
        const uint32_t x = word(i / 15), y = word(i % 225 < 15 && i < 225 ? i % 15 : 99);
        const float    u = (float)x * R_2POW32_INV + R_2POW32_INV;
        const float    v = R_2POW32_INV_2PI + (float)y * R_2POW32_INV_2PI;
        float          g[2];
        box_muller_dd<false>(u, v, ((y >> 19) + 8u) & ~15u, g[0], g[1]);
        const float       hs = sqrtf(-2.0f * logf(u)), h[2] = {sinf(v) * hs, cosf(v) * hs};
        const long double S = sqrtl(-2.0L * logl((long double)u));
        const __float128  e[2] = {(__float128)(sinl((long double)v) * S), (__float128)(cosl((long double)v) * S)};
        for(int j = 0; j < 2; j++)
        {
            beyond += ulps<float, int32_t>(g[j], h[j]) > 2;
            worst = e[j] != 0 ? fmax(worst, error<float>(g[j], e[j])) : worst;
        }
    }
    printf("pair_f32 %ld %ld %ld\n", 2 * n, (long)(worst * 1e6), beyond);
    worst  = 0.0;
    beyond = 0;
    double host = 0.0;
    for(long i = 0; i < n; i++)
    {
        const uint32_t a = word(i), b = word(i / 15), c = word(i), d = word(i < 225 ? i % 15 : 99);
        double         g[2];
        normal_pair_double(a, b, c, d, g[0], g[1]);
        const uint64_t v1 = (uint64_t)a ^ ((uint64_t)b << 21), v2 = (uint64_t)c ^ ((uint64_t)d << 21);
        const double   u = R_2POW53_INV_DBL + (double)v1 * R_2POW53_INV_DBL;
        const double   t = (R_2POW53_INV_DBL * 2.0 + (double)v2 * (R_2POW53_INV_DBL * 2.0)) * R_PI_DBL;
        const double   hs = sqrt(-2.0 * log(u)), h[2] = {sin(t) * hs, cos(t) * hs};
        const __float128 S = sqrtq(-2 * logq((__float128)u));
        const __float128 e[2] = {sinq((__float128)t) * S, cosq((__float128)t) * S};
        for(int j = 0; j < 2; j++)
        {
            beyond += ulps<double, int64_t>(g[j], h[j]) > 2;
            if(e[j] != 0)
            {
                worst = fmax(worst, error<double>(g[j], e[j]));
                host  = fmax(host, error<double>(h[j], e[j]));
            }
        }
    }
    printf("pair_f64 %ld %ld %ld\nsteps_f64 %ld\n", 2 * n, (long)(worst * 1e6), beyond, (long)(host * 1e6));
    printf("special %d %d %d %d\n", logf_unit(1.0f) == 0.0f, expf_acc(-200.0f) == 0.0f, isinf(expf_acc(200.0f)),
           isnan(expf_acc(NAN)));
    return 0;
}
#endif
