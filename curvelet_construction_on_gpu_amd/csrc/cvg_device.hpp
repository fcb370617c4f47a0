// Device-side building blocks shared by the curvelet kernels (k_curvelets_direct,
// k_curvelets_generic) and the diagnostic kernels, so that what the diagnostics
// check is the arithmetic those run.  (k_curvelets decides on certified
// approximations of it; tests compare its rows with these kernels' and the oracle's.)
#ifndef CVG_DEVICE_HPP
#define CVG_DEVICE_HPP

#include <hip/hip_runtime.h>

#include "cvg_math.hpp"

namespace cvg {

// Direction class of a neighbour: 1 when dot(To2Pi(atan2(ny-ay, nx-ax)), theta_a)
// > 0 (forward run), 2 when < 0 (backward run), 0 otherwise
// (cpu_curvelet.hpp:459-461, curvelet_utils.hpp:58-69).
//
// The reference's dot is cos(phi - theta_a), phi = atan2(vy, vx), v = n - a,
// up to its evaluation errors (atan2, To2Pi, cos, sin within an ulp each, the
// products and the sum), below 2e-15 in all.  The projection p = vx cos_at +
// vy sin_at, from the correctly rounded cos/sin of theta_a, is within 6e-16 |v|
// of |v| cos(phi - theta_a).  So when |p| > 1e-12 |v| the two signs agree and
// the class is sign(p); only near-perpendicular neighbours evaluate the
// reference's expression.
__device__ inline int direction_class(double ax, double ay, double cos_at, double sin_at, double nx, double ny,
                                      const double *sc_tab, const double *at_tab)
{
    const double vx = nx - ax, vy = ny - ay;
    const double p = vx * cos_at + vy * sin_at;
    if (fabs(p) > 1e-12 * sqrt(vx * vx + vy * vy)) return p > 0 ? 1 : 2;
    const double dir = wrap_two_pi(cr_atan2(vy, vx, at_tab));
    double sd, cd;
    cr_sincos(dir, sc_tab, &sd, &cd);
    const double dot = cd * cos_at + sd * sin_at;
    return dot > 0 ? 1 : (dot < 0 ? 2 : 0);
}

// One grid cell of the circular-arc bundle transport (Prop. 4),
// compute_curve_bundle's loop body (cpu_curvelet.hpp:697-751 for branch A,
// :762-806 for branch B), starting from [-max_k, max_k].  Operand order and
// rounding points are the reference's; the updates use the reference's
// compare-and-assign, which ignores NaN candidates.  The branches differ in
// powers of two on both sides of the curvature fraction, in the sign that an
// exactly zero denominator gets (:774 negates the sum), and in which of
// theta_n -+ dt bounds which side (branch A: theta_n - dt the lower).
//   DX, DY, DX2, DY2     n - a negated, and the squares (:646-649)
//   ox                   delta_x2 of the cell's row i
//   s2, c2               sin/cos(T2t), T2t = theta_a + delta_t2
//   s0, cx0, sy0         the lower constraint's angle T0: sin(T2t - T0), DX cos T0, DY sin T0 (:728-733)
//   s1, cx1, sy1         the upper's
__device__ inline void bundle_cell(double DX, double DY, double DX2, double DY2, bool branch_a, double ox, double s2,
                                   double c2, double s0, double cx0, double sy0, double s1, double cx1, double sy1,
                                   double dx, double dx2, double max_k, double &lo, double &hi)
{
    const double tt = s2 * DX - c2 * DY;  // :705
    const double ttm = tt - ox;
    const double u = 2.0 * ox * tt - DX2 - DY2 + dx2 - ox * ox;
    const double den = branch_a ? 0.0 - u : -u / 2.0;
    const double f = branch_a ? 2.0 : 1.0;
    const double kx0 = f * (ttm - dx) / den, kx1 = f * (ttm + dx) / den;
    const double kt0 = s0 / (-s0 * ox + cx0 + sy0), kt1 = s1 / (-s1 * ox + cx1 + sy1);
    lo = -max_k;
    hi = max_k;
    if (lo < kx0) lo = kx0;
    if (lo < kt0) lo = kt0;
    if (hi > kx1) hi = kx1;
    if (hi > kt1) hi = kt1;
}

}  // namespace cvg

#endif
