// Reciprocals, reciprocal square roots and what the kernels form from them,
// refined from estimates of 2^-20 or better. Est supplies the estimates:
// Est::rcp(x) ~ 1 / x, Est::rsq(x) ~ 1 / sqrt(x).
#pragma once
#include <cmath>
#include "hostdev.hpp"

namespace dmhm {

// 1 / x and 1 / sqrt(x) by two Newton steps each: a shorter dependent chain
// than IEEE division and square root, to rounding (u = 2^-53: 1.01 u and 2 u).
template <typename Est>
DMHM_HD double refined_rcp(double x)
{
    double r = Est::rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}
template <typename Est>
DMHM_HD double refined_rsq(double x)
{
    double y = Est::rsq(x);
    y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
    return fma(0.5 * y, fma(-x * y, y, 1.0), y);
}

// sqrt(x) for x > 0 from y, its refined reciprocal: x y is off by 3 u, the
// residual x - s^2, exact to its rounding, takes that back to one rounding.
DMHM_HD double refined_sqrt(double x, double y)
{
    const double s = x * y;
    return fma(fma(-s, s, x), 0.5 * y, s);
}

// Householder reflector I - tau v v^T, v = (1, scale x), of a column (alpha, x)
// of squared norm n2 = alpha^2 + x^T x: beta = -sgn(alpha) |column| (what it
// makes of alpha), tau = (beta - alpha) / beta, scale = 1 / (alpha - beta).
template <typename Est>
DMHM_HD void householder(double alpha, double n2, double& tau, double& scale, double& beta)
{
    const double rs = refined_rsq<Est>(n2), nrm = refined_sqrt(n2, rs);
    beta = -copysign(nrm, alpha);
    tau = fma(fabs(alpha), rs, 1.0);
    scale = copysign(refined_rcp<Est>(fabs(alpha) + nrm), alpha);
}

// Rotation (c, s) of a column pair with squared norms al, be and inner
// product ga that makes the pair orthogonal: t = tan(theta) is the root of
// t^2 + 2 zeta t - 1 = 0 of smaller magnitude, zeta = (be - al) / (2 ga),
// written as t = sgn(d) g / (|d| + sqrt(d^2 + g^2)) with d = be - al and
// g = 2 ga. t does not change when d and g are scaled together, so both are
// scaled by an estimate of 1 / max(|d|, |g|) first (no overflow or underflow
// in the squares). c = 1 / sqrt(1 + t^2), s = c t.
// (With one Newton step per estimate t keeps 46 bits. On random factors of
// 20 and 36 columns the cosines left were up to 1.6e-15 and 1.2e-14, against
// 1.0e-15 and 1.1e-15.)
template <typename Est>
DMHM_HD void jacobi_rotation(double al, double be, double ga, double& cs, double& sn)
{
    const double d0 = be - al, g0 = 2.0 * ga;
    const double rm = Est::rcp(fmax(fabs(d0), fabs(g0)));
    const double dd = d0 * rm, gg = g0 * rm;
    const double h = fma(dd, dd, gg * gg);
    const double den = fabs(dd) + h * refined_rsq<Est>(h);
    const double t = (dd >= 0.0 ? gg : -gg) * refined_rcp<Est>(den);
    cs = refined_rsq<Est>(fma(t, t, 1.0));
    sn = cs * t;
}

} // namespace dmhm
