// Host check of hamr_arith.h's Div at the ends of the exponent range, with the gfx950
// builtins it uses restated: the reciprocal estimate as 1/b cut to 22 bits, div_fixup
// as the selection of special quotients and, as the hardware has it, an infinity of
// the quotient's sign for a NaN between finite operands.
//  - numerators from 2^-969, divisors above 2^-1024: the IEEE quotient bit for bit,
//    overflowing and underflowing ones among them;
//  - smaller numerators: within one unit in the last place;
//  - divisors of 2^-1024 or less: an infinity of the quotient's sign;
//  - sixth: the IEEE quotient from 2^-969, NaN for an infinity.
// Exit status 0 when they hold.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

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
    if (!std::isfinite(a) || !std::isfinite(d) || a == 0. || d == 0.) return a / d;
    if (q == q) return q;
    return std::signbit(a) != std::signbit(d) ? -HUGE_VAL : HUGE_VAL;
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

int main()
{
    std::mt19937_64 g(12);
    std::uniform_real_distribution<double> U(1., 2.);
    const double inf = std::numeric_limits<double>::infinity();
    // +-1.x 2^e, the power itself among them
    auto num = [&](int e, int i) { return (i & 1 ? -1. : 1.) * std::ldexp(i & 2 ? 1. : U(g), e); };
    const int ends[] = {-1074, -1060, -1040, -1025, -1024, -1023, -1022, -1021, -1000, -970, -969, -968, -600, -500, -60, 0,
                        60, 500, 600, 960, 1000, 1019, 1020, 1021, 1022, 1023};
    for (int ea : ends)
        for (int ed : ends)
            for (int i = 0; i < 4000; i++) {
                const double a = num(ea, i), d = num(ed, i >> 2), q = a / d, r = hamr::Div<double>(d)(a);
                bool ok;
                if (std::fabs(d) <= std::ldexp(1., -1024)) ok = r == std::copysign(inf, q);
                else if (std::fabs(a) >= std::ldexp(1., -969)) ok = r == q;
                else ok = std::fabs(r - q) <= std::nextafter(std::fabs(q), inf) - std::fabs(q);
                if (!ok) return printf("%a / %a = %a, got %a\n", a, d, q, r), 1;
            }
    for (int ea : ends)
        for (int i = 0; ea >= -969 && i < 4000; i++) {
            const double a = num(ea, i);
            if (hamr::sixth(a) != a / 6.) return printf("%a / 6\n", a), 1;
        }
    return hamr::sixth(inf) != hamr::sixth(inf) ? 0 : (printf("sixth(inf)\n"), 1);
}
