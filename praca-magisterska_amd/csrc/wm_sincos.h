// sin and cos of the fill's phase arguments k R (0 <= x < kSinCosMax).
//
// Cody & Waite argument reduction (W. J. Cody, W. Waite, "Software Manual for
// the Elementary Functions", 1980): n = rint(x 2/pi), r = x - n pi/2 with
// pi/2 split into three parts, P1 and P2 of 33 significant bits (so n P1 and
// n P2 are exact for n < 2^20) and P3 the remainder, each subtracted with a
// fused multiply-add; then sin r and cos r on |r| <= pi/4 (a little beyond
// after rounding n) from minimax polynomials (this project's own fit: weighted
// least squares in 80-bit arithmetic, reweighted to a level error; with the
// coefficients rounded to double the errors relative to the result are 6.0e-18 and
// 1.5e-18, a twentieth of an ulp at most: the rounding of -1/6 decides the sine's, and the
// Taylor sums through r^17 and r^16 used before are no better, 6.4e-18 and 1.6e-18,
// with one more term each), and the quadrant n mod 4.
// Every rounding is written out, so host and device builds give the same bits.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define WM_HD __host__ __device__
#else
#define WM_HD
#endif

namespace wm {

constexpr double kSinCosMax = 1.6e6;  // below 2^20 pi/2: n P1 and n P2 stay exact

// The constants, as values that a kernel can keep in registers of its choice.
struct SinCosConsts {
    double two_over_pi = 0.6366197723675814;
    double p1 = 1.5707963267341256, p2 = 6.077100506303966e-11, p3 = 2.0222662487959506e-21;
    // sin r = r + r^3 (s[6] + r^2 (s[5] + ...)),  cos r = 1 + r^2 (-1/2 + r^2 (c[5] + r^2 (c[4] + ...)))
    double s[7] = {-7.5786380750307477e-13,
                   1.6058359290223325e-10,
                   -2.5052104800183583e-08,
                   2.7557319213547918e-06,
                   -0.00019841269841253486,
                   0.0083333333333333211,
                   -0.16666666666666666};
    double c[6] = {-1.1358412519525422e-11,
                   2.0875698350458964e-09,
                   -2.7557314160173976e-07,
                   2.4801587288782315e-05,
                   -0.0013888888888872939,
                   0.041666666666666595};
};

WM_HD inline void sincos_phase(double x, double &s, double &c, const SinCosConsts &k = SinCosConsts())
{
    const double n = rint(x * k.two_over_pi);
    double r = fma(-n, k.p1, x);
    r = fma(-n, k.p2, r);
    r = fma(-n, k.p3, r);
    const double r2 = r * r;
    double ps = k.s[0], pc = k.c[0];
    for (int i = 1; i < 7; ++i) ps = fma(ps, r2, k.s[i]);
    for (int i = 1; i < 6; ++i) pc = fma(pc, r2, k.c[i]);
    pc = fma(pc, r2, -0.5);
    const double sr = fma(r * r2, ps, r);
    const double cr = fma(r2, pc, 1.0);
    // quadrant q: (sin, cos) = (s, c), (c, -s), (-s, -c), (-c, s) for q = 0..3
    const int q = (int)n & 3;
    const double a = (q & 1) ? cr : sr, b = (q & 1) ? sr : cr;
    s = (q & 2) ? -a : a;
    c = ((q + 1) & 2) ? -b : b;
}

}  // namespace wm
