// hamr_arith.h -- division, reciprocal square root and power in the arithmetic R
// of a kernel.  HAMR_DEVICE_ARITH selects the device forms; a host program may
// set it with HD and the gfx950 builtins they use defined, to check them.
#pragma once

#include <cmath>

#if !defined(HAMR_DEVICE_ARITH) && defined(__HIP_DEVICE_COMPILE__)
#define HAMR_DEVICE_ARITH 1
#endif

namespace hamr {

// Division, reciprocal square root and power in the arithmetic of R: IEEE
// double operations for the FP64 step (the reference's), the hardware's
// single-precision reciprocal, reciprocal square root and exp2/log2 (about
// one ulp each) for the FP32 path.
template <class R> HD R dv(R a, R b) { return a / b; }
template <class R> HD R rsq(R a) { return R(1.) / sqrt(a); }
template <class R> HD R rpow(R a, R e) { return pow(a, e); }
#if HAMR_DEVICE_ARITH
template <> HD float dv<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
template <> HD float rsq<float>(float a) { return __builtin_amdgcn_rsqf(a); }
template <> HD float rpow<float>(float a, float e) { return __builtin_amdgcn_exp2f(e * __builtin_amdgcn_logf(a)); }
#endif

// Quotients by one divisor.  On the device in FP64, the reciprocal part of the
// division (hardware estimate, two Newton steps) is formed once per divisor,
// and each quotient takes the last step of the IEEE division on it (product,
// residual, correction, special values): 4 instructions instead of 11 with a
// quarter-rate estimate among them.  These are the operations the compiler's
// own division performs when it does not rescale its operands, so for a numerator
// from 2^-969 on and a divisor above 2^-1024 the result is the same correctly
// rounded quotient, an overflowing one the same infinity (div_fixup makes it of the
// NaN that the residual then is); a smaller numerator gives it within one unit in
// the last place.  A divisor of 2^-1024 or less, whose reciprocal overflows, gives
// an infinity also where the quotient is finite: no divisor of the step comes near
// (densities, enthalpies, Lorentz factors, wave speeds with kSMALL added, metric
// determinants).  Zeros, infinities and NaNs divide as IEEE.
// The FP64 flux kernel forms 31 quotients by 10 divisors a face, the update 60 by 17
// (9 by 6 of them in every Newton iteration).  In FP32 the quotient is a * rcp(b),
// as dv.
template <class R> struct Div {
    R d;
    HD explicit Div(R b) : d(b) {}
    HD Div(R b, R) : d(b) {}  // with the reciprocal formed earlier
    HD R recip() const { return R(0.); }
    HD R operator()(R a) const { return dv(a, d); }
};
#if HAMR_DEVICE_ARITH
template <> struct Div<double> {
    double d, y;
    HD explicit Div(double b) : d(b)
    {
        y = __builtin_amdgcn_rcp(b);
        y = fma(y, fma(-b, y, 1.), y);
        y = fma(y, fma(-b, y, 1.), y);
    }
    HD Div(double b, double r) : d(b), y(r) {}
    HD double recip() const { return y; }
    HD double operator()(double a) const
    {
        const double q = a * y;
        return __builtin_amdgcn_div_fixup(fma(fma(-d, q, a), y, q), d, a);
    }
};
#endif

// a / 6, 21 of them a face: Div's quotient by a constant reciprocal, without its
// treatment of infinite a (the quotient is then NaN, not infinite).
template <class R> HD R sixth(R a) { return Div<R>(R(6.))(a); }
#if HAMR_DEVICE_ARITH
template <> HD double sixth<double>(double a)
{
    const double y = 1. / 6., q = a * y;
    return fma(fma(-6., q, a), y, q);
}
#endif

#if HAMR_DEVICE_ARITH
// x^e in FP64 on the device, for the entropy of a state (x = rho).  The library
// pow is 226 VALU instructions, 18% of the FP64 flux kernel, for two per face;
// this one is 78.  log2 x = k + (2 / ln 2) atanh(s), s = (m - 1) / (m + 1), x = m
// 2^k with m in [sqrt(1/2), sqrt(2)), in two words (s with its residual, the
// series (atanh(s) - s) / s^3 to 1e-18); 2^(e log2 x) by its nearest integer and
// a polynomial of degree 11 in the rest, again with its rounding carried along.
// Coefficients: interpolation at the Chebyshev nodes of [0, (3 - 2 sqrt 2)^2]
// and [-1/2, 1/2] in 60-digit arithmetic.  Largest error on 4e6 x in 1e-13 ..
// 1e13 for e = -13/9, -4/3, -5/3: 0.74 units in the last place (rms 0.290);
// the device library's pow: 1.31 (rms 0.416).
// Special x as pow's: 0 and infinity take the exponent -+2^14 (2^(e log2 x) then
// overflows or vanishes by the sign of e), a negative x gives NaN, or +-|x|^e for
// a whole e, by selects rather than a branch (a branch to the library's pow cost
// the flux kernels 260 bytes of spilled registers).
template <> HD double rpow<double>(double x, double e)
{
    const double ax = fabs(x);
    const bool edge = ax == 0. || ax == __builtin_inf();
    double m = edge ? 1.0 : __builtin_amdgcn_frexp_mant(ax);
    const bool low = m < 0.70710678118654752440;
    int k = __builtin_amdgcn_frexp_exp(ax) - (low ? 1 : 0);
    if (edge) k = ax > 1. ? 1 << 14 : -(1 << 14);
    m = low ? m + m : m;
    const double u = m - 1.0, v = m + 1.0, vl = m - (v - 1.0);
    const Div<double> D(v);
    const double s = u * D.y;
    const double sl = fma(-s, vl, fma(-s, v, u)) * D.y, z = s * s;
    double p = 0x1.0c039c49989c6p-4;
    p = fma(p, z, 0x1.0fbe95d716020p-4);
    p = fma(p, z, 0x1.3b1c355a8f7a2p-4);
    p = fma(p, z, 0x1.745cf9048dd95p-4);
    p = fma(p, z, 0x1.c71c720159177p-4);
    p = fma(p, z, 0x1.2492492476cccp-3);
    p = fma(p, z, 0x1.9999999999a38p-3);
    p = fma(p, z, 0x1.5555555555555p-2);
    const double w = fma(s * z, p, sl);
    const double ch = 0x1.71547652b82fep+1, cl = 0x1.777d0ffda0d24p-55;  // 2 / ln 2
    const double a = s * ch;
    const double al = fma(w, ch, fma(s, cl, fma(s, ch, -a)));
    const double hi = (double)k + a, lo = (a - (hi - (double)k)) + al;  // |a| <= 1/2: exact two-word sum
    const double E = e * hi, El = fma(e, lo, fma(e, hi, -E));
    const double n = rint(E), f0 = E - n, f = f0 + El, fl = El - (f - f0);
    double q = 0x1.e9d3fe3952179p-32;
    q = fma(q, f, 0x1.e6063f7217bc6p-28);
    q = fma(q, f, 0x1.b524fae627834p-24);
    q = fma(q, f, 0x1.62bfd47773353p-20);
    q = fma(q, f, 0x1.ffcbfc670dcd4p-17);
    q = fma(q, f, 0x1.430913096fd9fp-13);
    q = fma(q, f, 0x1.5d87fe78a5276p-10);
    q = fma(q, f, 0x1.3b2ab6fba1ddap-7);
    q = fma(q, f, 0x1.c6b08d704a0c2p-5);
    q = fma(q, f, 0x1.ebfbdff82c598p-3);
    const double L = 0x1.62e42fefa39efp-1, Ll = 0x1.abc9e3b39803fp-56;  // ln 2
    const double b = f * q, g = L + b, gl = ((L - g) + b) + Ll;
    const double t = f * g, tl = fma(fl, L, fma(f, gl, fma(f, g, -t)));
    const double r = 1.0 + t;
    const double v2 = ldexp(r + (((1.0 - r) + t) + tl), (int)n);
    const double neg = e == rint(e) ? (0.5 * e == rint(0.5 * e) ? 1.0 : -1.0) : __builtin_nan("");
    return x < 0. ? neg * v2 : v2;
}
#endif

}  // namespace hamr
