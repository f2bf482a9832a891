// Trigonometry of the integrator, in fp64 with one rounding to fp32.
//
// The arguments are bounded (angles of warps within [-2 pi, 2 pi], unit directions), so the general library
// functions' wide argument reduction and extended-precision branches are not needed: they are what held the
// shading kernels' registers. Argument reduction by pi/2 in two parts with fused multiply-adds, then Taylor
// polynomials on [-pi/4, pi/4]; the arctangent is reduced to |t| <= tan(pi/8) and evaluated with a polynomial
// that interpolates it at 12 Chebyshev nodes (error below 1.5e-18, a thirtieth of a unit). Each fp64 value is within
// 2 units in its last place, the arccosine's, which comes from an arctangent of a square root, within 3 (measured
// against numpy: tests/test_trig_cpu.py), so the fp32 results are the correctly rounded ones except with a
// probability of about 2^-27 per call.
#pragma once

#include <stdint.h>

namespace phd {

// sin and cos of x, |x| <= 64.
PH_DEV void sincos64(double x, double* s, double* c) {
    const double n = __builtin_rint(x * 0x1.45f306dc9c883p-1);
    double r = __builtin_fma(-n, 0x1.921fb54442d18p+0, x);
    r = __builtin_fma(-n, 0x1.1a62633145c07p-54, r);
    const double z = r * r;
    double p = __builtin_fma(z, -1.0 / 1307674368000.0, 1.0 / 6227020800.0);
    p = __builtin_fma(z, p, -1.0 / 39916800.0);
    p = __builtin_fma(z, p, 1.0 / 362880.0);
    p = __builtin_fma(z, p, -1.0 / 5040.0);
    p = __builtin_fma(z, p, 1.0 / 120.0);
    p = __builtin_fma(z, p, -1.0 / 6.0);
    const double sn = __builtin_fma(r * z, p, r);
    double q = __builtin_fma(z, 1.0 / 20922789888000.0, -1.0 / 87178291200.0);
    q = __builtin_fma(z, q, 1.0 / 479001600.0);
    q = __builtin_fma(z, q, -1.0 / 3628800.0);
    q = __builtin_fma(z, q, 1.0 / 40320.0);
    q = __builtin_fma(z, q, -1.0 / 720.0);
    q = __builtin_fma(z, q, 1.0 / 24.0);
    q = __builtin_fma(z, q, -0.5);
    const double cs = __builtin_fma(z, q, 1.0);
    const int k = int(n);
    const double a = (k & 1) ? cs : sn, b = (k & 1) ? sn : cs;
    *s = (k & 2) ? -a : a;
    *c = ((k + 1) & 2) ? -b : b;
}

// atan2(y, x) for finite or NaN arguments whose larger magnitude is neither denormal nor huge, and for zeros.
PH_DEV double atan2_64(double y, double x) {
    const double ay = __builtin_fabs(y), ax = __builtin_fabs(x);
    const bool steep = ay > ax;
    const double hi = steep ? ay : ax, lo = steep ? ax : ay;
    const bool upper = lo > 0.41421356237309503 * hi;  // atan(lo / hi) = pi/4 + atan((lo - hi) / (lo + hi))
    const double num = upper ? lo - hi : lo, den = upper ? lo + hi : (hi == 0.0 ? 1.0 : hi);
    const double t = num / den, z = t * t;
    double p = 0x1.0acbaedf84569p-6;
    p = __builtin_fma(z, p, -0x1.1b302522803dcp-5);
    p = __builtin_fma(z, p, 0x1.74dc632cec5e9p-5);
    p = __builtin_fma(z, p, -0x1.ac7a3e94221b0p-5);
    p = __builtin_fma(z, p, 0x1.e19a0757950b1p-5);
    p = __builtin_fma(z, p, -0x1.110e8771e02b1p-4);
    p = __builtin_fma(z, p, 0x1.3b1392d01a746p-4);
    p = __builtin_fma(z, p, -0x1.745d165d8a943p-4);
    p = __builtin_fma(z, p, 0x1.c71c71c301fcdp-4);
    p = __builtin_fma(z, p, -0x1.249249248d7a0p-3);
    p = __builtin_fma(z, p, 0x1.9999999999953p-3);
    p = __builtin_fma(z, p, -0x1.5555555555555p-2);
    double a = __builtin_fma(t * z, p, t);
    // The lower parts of pi/4, pi/2 and pi keep the sums within an ulp.
    if (upper) a = 0x1.921fb54442d18p-1 + (a + 0x1.1a62633145c07p-55);
    if (steep) a = 0x1.921fb54442d18p+0 - (a - 0x1.1a62633145c07p-54);
    if (__builtin_signbit(x)) a = 0x1.921fb54442d18p+1 - (a - 0x1.1a62633145c07p-53);
    return __builtin_copysign(a, y);
}

PH_DEV void sincos_cr(float x, float* s, float* c) {
    double sd, cd;
    sincos64(double(x), &sd, &cd);
    *s = float(sd);
    *c = float(cd);
}
PH_DEV float atan2_cr(float y, float x) { return float(atan2_64(double(y), double(x))); }
// x in [-1, 1].
PH_DEV double acos64(double x) { return atan2_64(__builtin_sqrt((1.0 - x) * (1.0 + x)), x); }
PH_DEV float acos_cr(float x) { return float(acos64(double(x))); }

}  // namespace phd
