// Host check of the device forms of hamr_arith.h, with the gfx950 builtins they
// use restated: the reciprocal estimate as 1/b cut to 22 bits (the hardware's is
// at least that good), div_fixup as the selection of special quotients.
//  - Div: the IEEE quotient bit for bit where no intermediate leaves the normal
//    range, within one unit in the last place below 2^-969, the IEEE results for
//    zeros, infinities and NaNs;
//  - rpow: within 1 unit in the last place of the 113-bit power (the two-word
//    logarithm and exponential leave at most 0.25 beyond the final rounding's
//    1/2), pow's results for special arguments.
// Exit status 0 when they hold.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

#include <quadmath.h>

#define HD inline
#define HAMR_DEVICE_ARITH 1
static double __builtin_amdgcn_rcp(double b)
{
    double y = 1.0 / b;
    uint64_t u;
    std::memcpy(&u, &y, 8);
    if (std::isfinite(y)) u &= ~((1ull << 31) - 1);
    std::memcpy(&y, &u, 8);
    return y;
}
static double __builtin_amdgcn_div_fixup(double q, double d, double a)
{
    const bool special = !std::isfinite(a) || !std::isfinite(d) || a == 0. || d == 0.;
    return special ? a / d : q;
}
static float __builtin_amdgcn_rcpf(float b) { return 1.f / b; }
static float __builtin_amdgcn_rsqf(float b) { return 1.f / std::sqrt(b); }
static float __builtin_amdgcn_exp2f(float b) { return std::exp2(b); }
static float __builtin_amdgcn_logf(float b) { return std::log2(b); }
static int __builtin_amdgcn_frexp_exp(double x)
{
    int k = 0;
    if (std::isfinite(x)) std::frexp(x, &k);
    return k;
}
static double __builtin_amdgcn_frexp_mant(double x)
{
    int k;
    return std::frexp(x, &k);
}
#include "hamr_arith.h"

static bool same(double a, double b) { return (a != a && b != b) || a == b; }

int main()
{
    std::mt19937_64 g(11);
    std::uniform_real_distribution<double> U(0., 1.);
    const double inf = std::numeric_limits<double>::infinity(), nan = std::numeric_limits<double>::quiet_NaN();
    auto num = [&](double span) { return (U(g) < 0.5 ? -1. : 1.) * std::ldexp(0.5 + U(g), (int)((2. * U(g) - 1.) * span)); };
    long bad = 0;
    for (long i = 0; i < 4000000; i++) {
        double a = num(i & 1 ? 8. : 400.), d = num(i & 1 ? 8. : 400.);
        if (i % 7 == 0) d = 6.0;
        if (i % 11 == 0) a = std::nextafter(d * (double)(1 + i % 13), i & 2 ? inf : -inf);
        if (hamr::Div<double>(d)(a) != a / d) bad++;
    }
    if (bad) return printf("Div: %ld quotients differ from IEEE division\n", bad), 1;
    for (long i = 0; i < 400000; i++) {
        const double d = num(8.), a = std::ldexp(num(8.), -1010), q = a / d, r = hamr::Div<double>(d)(a);
        if (std::fabs(r - q) > std::fabs(std::nextafter(q, inf) - q)) return printf("Div: %a / %a = %a, got %a\n", a, d, q, r), 1;
    }
    const double sp[] = {0., -0., 1., -3., inf, -inf, nan};
    for (double a : sp)
        for (double d : sp)
            if (!same(hamr::Div<double>(d)(a), a / d)) return printf("Div: %g / %g\n", a, d), 1;

    double worst = 0.;
    const double es[] = {-13. / 9., -4. / 3., -5. / 3., -1.4, 4. / 9., -2., 0.75};
    for (double e : es)
        for (long i = 0; i < 300000; i++) {
            const double x = (i & 1) ? std::exp((2. * U(g) - 1.) * (i & 2 ? 30. : 250.)) : 0.5 + 1.5 * U(g);
            const double r = hamr::rpow(x, e);
            const __float128 t = powq(x, e);
            const double ulp = std::ldexp(1., std::ilogb((double)t) - 52);
            worst = std::fmax(worst, std::fabs((double)((r - t) / ulp)));
        }
    printf("rpow: largest error %.3f units in the last place\n", worst);
    if (!(worst < 1.0)) return 1;
    for (double e : es)
        for (double x : {0., inf, nan, -2., -0.5, 1., 4.9e-324, 2.2e-308, 1.7e308}) {
            const double r = hamr::rpow(x, e), t = std::pow(x, e);
            if (!same(r, t) && !(std::fabs(r - t) <= 2.3e-16 * std::fabs(t)))
                return printf("rpow(%g, %g) = %a, pow %a\n", x, e, r, t), 1;
        }
    return 0;
}
