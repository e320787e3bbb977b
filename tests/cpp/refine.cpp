// refine.hpp on the host, with estimates as poor as the hardware's may be
// (relative error 2^-23 either way), against long double. u = 2^-53. Exits with
// 1 and a line at the first value outside its bound.
#include <cstdio>
#include <cstdlib>
#include <random>
#include "refine.hpp"

static int side = 0;            // which way the estimates err
struct Est {
    static double off(double v) { side = (side + 1) & 3; return v * (1.0 + ((side & 1) ? 1.0 : -1.0) * std::ldexp(1.0, -23)); }
    static double rcp(double x) { return off(1.0 / x); }
    static double rsq(double x) { return off(1.0 / std::sqrt(x)); }
};

static const long double U = 1.0L / 9007199254740992.0L;
static void bound(const char* what, long double got, long double want, double units, double x)
{
    if (fabsl(got - want) <= units * U * fabsl(want)) return;
    std::printf("%s: %.2f u at %a\n", what, (double)(fabsl(got - want) / (U * fabsl(want))), x);
    std::exit(1);
}

int main()
{
    std::mt19937_64 g(1);
    std::uniform_real_distribution<double> mant(1.0, 2.0), unit(-1.0, 1.0);
    std::uniform_int_distribution<int> expo(-300, 300), near(-30, 30);
    for (int i = 0; i < 1000000; ++i) {
        const double x = std::ldexp(mant(g), expo(g));
        // One rounding; the last step's own error is below 2^-60.
        bound("rcp", dmhm::refined_rcp<Est>(x), 1.0L / x, 1.01, x);
        // Half of the rounding of x y, half of that of its square, the last one.
        bound("rsq", dmhm::refined_rsq<Est>(x), 1.0L / sqrtl(x), 2.01, x);
        // The residual's correction leaves the rounding of the sum alone.
        bound("sqrt", dmhm::refined_sqrt(x, dmhm::refined_rsq<Est>(x)), sqrtl(x), 1.01, x);
        // Reflector: beta one rounding; tau 2 u of a term of at most half of it
        // and one rounding; scale beta's, the sum's and the reciprocal's.
        const double alpha = std::sqrt(x) * unit(g);
        double tau, scale, beta;
        dmhm::householder<Est>(alpha, x, tau, scale, beta);
        const long double b = -copysignl(sqrtl(x), alpha);
        bound("beta", beta, b, 1.01, x);
        bound("tau", tau, (b - alpha) / b, 2.02, x);
        bound("scale", scale, 1.0L / (alpha - b), 3.03, x);
        // tan of the rotation: d (1), its scaling and g's (2), h (2), its root
        // (2 + 1), the sum (1), the reciprocal (1), the product (1).
        const double al = std::ldexp(mant(g), near(g)), be = std::ldexp(mant(g), near(g));
        const double ga = unit(g) * std::sqrt(al * be);
        double c, s;
        dmhm::jacobi_rotation<Est>(al, be, ga, c, s);
        const long double d = (long double)be - al, gg = 2.0L * ga;
        const long double t = (d >= 0 ? gg : -gg) / (fabsl(d) + sqrtl(d * d + gg * gg));
        // sn = c t adds one rounding, the quotient taken here none.
        bound("tan", (long double)s / c, t, 12, ga);
        bound("c^2 + s^2", (long double)c * c + (long double)s * s, 1.0L, 8, ga);
    }
    std::puts("ok");
    return 0;
}
