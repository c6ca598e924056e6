/* Host twin of the normal and log-normal transforms' functions
 * (include/rocrand/rocrand_amd_math.h: logf_unit, sincosf_unit, expf_acc, box_muller_dd,
 * normal_pair_double): the same source compiled for the host, checked against long double
 * and quad precision and against the reference's steps over this libm.  The device's
 * reciprocal square roots are emulated to their precision (2^-24).
 *
 * usage: normal_twin N
 * prints NAME COUNT VALUES  for the float functions' results that are not the correctly
 * rounded ones, and  NAME VALUES MAX_ERR_MICROULP BEYOND_2ULP_OF_LIBM  and the MAX_ERR_MICROULP
 * of the reference's steps over this libm for the pairs.
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
// words at the ends of their range and next to the angle tables' boundaries (odd multiples
// of 2^22 for the float pair, of 2^23 for the others), then random; the first EDGES^2
// pairs are all pairs of the edges
static const uint32_t edge[] = {0u,          1u,          0x1fffffu,   0x200000u,   0x3fffffu,   0x400000u,   0x400001u,
                                0x7fffffu,   0x800000u,   0x3fffffffu, 0x40000000u, 0x7fbfffffu, 0x7fc00000u, 0x7fffffffu,
                                0x80000000u, 0x803fffffu, 0x80400000u, 0xbfffffffu, 0xffbfffffu, 0xffc00000u, 0xffffff7fu,
                                0xffffff80u, 0xfffffffeu, 0xffffffffu};
constexpr long        EDGES  = sizeof(edge) / sizeof(edge[0]);
static uint32_t word(long i)
{
    return i < EDGES ? edge[i] : (uint32_t)(next64() >> 13);
}
static uint32_t word_x(long i) { return word(i < EDGES * EDGES ? i / EDGES : EDGES); }
static uint32_t word_y(long i) { return word(i < EDGES * EDGES ? i % EDGES : EDGES); }

// The float pair: rows as for the double pair below; a sign that differs from the steps'
// (a radius of -0 keeps its sign) counts as beyond.
template<class F>
static void pair_f32_row(const char* name, long n, F uv)
{
    double worst = 0.0, host = 0.0;
    long   beyond = 0;
    for(long i = 0; i < n; i++)
    {
        float    u, v, g[2];
        uint32_t qoff;
        uv(word_x(i), word_y(i), u, v, qoff);
        box_muller_dd<false>(u, v, qoff, g[0], g[1]);
        const float       hs = sqrtf(-2.0f * logf(u)), h[2] = {sinf(v) * hs, cosf(v) * hs};
        const long double S = sqrtl(-2.0L * logl((long double)u));
        const __float128  e[2] = {(__float128)(sinl((long double)v) * S), (__float128)(cosl((long double)v) * S)};
        for(int j = 0; j < 2; j++)
        {
            beyond += ulps<float, int32_t>(g[j], h[j]) > 2 || !signbit(g[j]) != !signbit(h[j]);
            if(e[j] != 0)
            {
                worst = fmax(worst, error<float>(g[j], e[j]));
                host  = fmax(host, error<float>(h[j], e[j]));
            }
        }
    }
    printf("%s %ld %ld %ld %ld\n", name, 2 * n, (long)(worst * 1e6), beyond, (long)(host * 1e6));
}
// mrg_box_muller's float uniform and angle of values in [1, m1]
template<int MRG>
static void mrg_uv(uint32_t x, uint32_t y, float& u, float& v, uint32_t& qoff)
{
    constexpr uint64_t m1 = MRG == 32 ? 4294967087ull : 2147483647ull;
    x = x == 0xffffffffu ? (uint32_t)m1 : 1u + (uint32_t)((MRG == 32 ? x : x >> 1) % m1); // u = 1 among them
    y = 1u + (uint32_t)((MRG == 32 ? y : y >> 1) % m1);
    u    = (float)((double)x * mrg_consts<MRG>::norm);
    v    = (float)((double)y * mrg_consts<MRG>::norm) * R_2PI;
    qoff = ((y >> (MRG == 32 ? 19 : 18)) + 8u) & ~15u;
}

// The double pair at angle t, radius uniform u: worst error in ulp of exact and, in `beyond`,
// the values more than 2 ulp from the reference's steps over this libm, whose own worst
// error goes to `host`.
static void pair_check(double u, double t, const double (&g)[2], double& worst, long& beyond, double& host)
{
    const double     hs = sqrt(-2.0 * log(u)), h[2] = {sin(t) * hs, cos(t) * hs};
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
static void pair_words(uint32_t a, uint32_t b, uint32_t c, uint32_t d, double& worst, long& beyond, double& host)
{
    double g[2];
    normal_pair_double(a, b, c, d, g[0], g[1]);
    const uint64_t v1 = (uint64_t)a ^ ((uint64_t)b << 21), v2 = (uint64_t)c ^ ((uint64_t)d << 21);
    const double   u = R_2POW53_INV_DBL + (double)v1 * R_2POW53_INV_DBL;
    const double   t = (R_2POW53_INV_DBL * 2.0 + (double)v2 * (R_2POW53_INV_DBL * 2.0)) * R_PI_DBL;
    pair_check(u, t, g, worst, beyond, host);
}
template<int MRG>
static void pair_mrg(uint32_t x, uint32_t y, double& worst, long& beyond, double& host)
{
    double g[2];
    mrg_normal_pair_double<MRG>(x, y, g[0], g[1]);
    const float u = (float)((double)x * mrg_consts<MRG>::norm), v = (float)((double)y * mrg_consts<MRG>::norm);
    pair_check((double)u, (double)v * 2.0 * R_PI_DBL, g, worst, beyond, host);
}

// The double pair next to the multiples of a quarter turn, where the sine or cosine is as
// small as the angle's own rounding: every w = (v2 + 1) 2^-52 within 256 steps of 0, 1/2,
// 1, 3/2 and 2, and the MRG words next to those that round to these (a float angle is
// exactly a quarter turn for a few hundred words), `n` radius words each.
template<class F>
static void quarter_row(const char* name, long count, F one)
{
    double worst = 0.0, host = 0.0;
    long   beyond = 0, total = 0;
    for(long i = 0; i < count; i++)
        total += 2 * one(i, worst, beyond, host);
    printf("%s %ld %ld %ld %ld\n", name, total, (long)(worst * 1e6), beyond, (long)(host * 1e6));
}
template<int MRG>
static void mrg_quarter_row(const char* name, int n)
{
    constexpr uint64_t m1 = MRG == 32 ? 4294967087ull : 2147483647ull;
    quarter_row(name, 5 * 601, [&](long i, double& worst, long& beyond, double& host) {
        const int64_t y = (int64_t)((i / 601) * ((m1 + 1) / 4)) + i % 601 - 300;
        if(y < 1 || y > (int64_t)m1)
            return 0;
        for(int k = 0; k < n; k++)
            pair_mrg<MRG>(k == 0 ? 1u : k == 1 ? (uint32_t)m1 : 1u + (uint32_t)(next64() % m1), (uint32_t)y, worst,
                          beyond, host);
        return n;
    });
}
static void quarter_rows(int n)
{
    quarter_row("quarter_words", 5 * 513, [&](long i, double& worst, long& beyond, double& host) {
        const int64_t v2 = (int64_t)(i / 513) * (1ll << 51) - 1 + i % 513 - 256;
        if(v2 < 0 || v2 >= 1ll << 53)
            return 0;
        const uint32_t d = (uint32_t)(v2 >> 32) << 11, c = (uint32_t)v2;
        for(int k = 0; k < n; k++)
        {
            const uint64_t x = k == 0 ? 0 : k == 1 ? ~0ull : next64();
            pair_words((uint32_t)x, (uint32_t)(x >> 32), c, d, worst, beyond, host);
        }
        return n;
    });
    mrg_quarter_row<32>("quarter_mrg32", n);
    mrg_quarter_row<31>("quarter_mrg31", n);
}

// log2 of the worst relative error of the doubles that are rounded to float, in hundredths
static void steps_row()
{
    double ws = 0.0, we = 0.0;
    auto   rel = [](double got, __float128 exact) { return (double)fabsq(((__float128)got - exact) / exact); };
    auto   angle = [&](uint32_t y) {
        const float v = R_2POW32_INV_2PI + (float)y * R_2POW32_INV_2PI;
        double      s, c;
        sincos_unit(v, ((y >> 20) + 8u) & ~15u, s, c);
        ws = fmax(ws, fmax(rel(s, sinq((__float128)v)), rel(c, cosq((__float128)v))));
    };
    for(long i = 0; i < 200000; i++)
        angle((uint32_t)(next64() >> 13));
    for(uint32_t q = 0; q < 4; q++) // next to the quarter turns, and the table's boundaries
        for(uint32_t k = 0; k < 2000; k++)
            angle((q << 30) + 256 * k), angle((q << 30) - 1 - 256 * k), angle((uint32_t)(next64() >> 13) & 0xff000000u | 0x00800000u);
    for(long i = 0; i < 400000; i++)
    {
        const float x = -105.0f + (float)i * (195.0f / 400000);
        we = fmax(we, rel(exp_acc(x), expq((__float128)x)));
    }
    printf("steps %ld %ld\n", (long)(100 * log2(ws)), (long)(100 * log2(we)));
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
    pair_f32_row("pair_f32", 5 * n, [](uint32_t x, uint32_t y, float& u, float& v, uint32_t& qoff) {
        u    = (float)x * R_2POW32_INV + R_2POW32_INV;
        v    = R_2POW32_INV_2PI + (float)y * R_2POW32_INV_2PI;
        qoff = ((y >> 19) + 8u) & ~15u;
    });
    pair_f32_row("pair_f32_mrg32", 5 * n, mrg_uv<32>);
    pair_f32_row("pair_f32_mrg31", 5 * n, mrg_uv<31>);
    double worst = 0.0, host = 0.0;
    long   beyond = 0;
    for(long i = 0; i < n; i++)
    {
        const uint32_t a = word(i), b = word_x(i), c = word(i), d = word_y(i);
        pair_words(a, b, c, d, worst, beyond, host);
    }
    printf("pair_f64 %ld %ld %ld %ld\n", 2 * n, (long)(worst * 1e6), beyond, (long)(host * 1e6));
    quarter_rows((int)(n / 4000));
    steps_row();
    printf("special %d %d %d %d\n", logf_unit(1.0f) == 0.0f, expf_acc(-200.0f) == 0.0f, isinf(expf_acc(200.0f)),
           isnan(expf_acc(NAN)));
    return 0;
}
#endif
