// fqsl_step.h -- the RKF45 step controller of the plain side tracers
// (TraceBlineAdaptive.cu:365-370) from estimates of a reciprocal square root and of
// a fifth root, with the results of the written expressions
//   scale = (tol / sqrt(e2) / 11.09)^0.2.
//
// FQSL_HD and FQSL_COLD are the includer's; on the device the estimates are
// instructions, the CPU tests pass their own.
#pragma once

#include <math.h>

namespace fqsl {

// tol / sqrt(e2) / 11.09, each operation rounded as the written expression rounds it,
// from r, which is 1 / sqrt(e2) within 2^-22: ~20 instructions instead of ~70.
// Goldschmidt's iteration takes sqrt(e2) and half its reciprocal to 2^-44, then each
// result is corrected by its exact remainder (a fused multiply-add) over a reciprocal
// good to a few 2^-53, which leaves the correctly rounded value (Markstein's method:
// the remainder of a value within one last place is exact, and a quotient by a
// constant needs that constant's correctly rounded reciprocal).  Holds where nothing
// under- or overflows: see step_is_plain.  (A step size is the product of all scales
// before it, and near the float floor of the error norm one last bit leads to other
// steps.)
FQSL_HD double scale_argument(double tol, double e2, double r) {
#if defined(__clang__)
#pragma clang fp contract(off)  // a product and its remainder are not fused
#endif
    double g = e2 * r, h = 0.5 * r;
    const double d = fma(-h, g, 0.5);
    g = fma(g, d, g);
    h = fma(h, d, h);
    g = fma(fma(-g, g, e2), h, g);
    g = fma(fma(-g, g, e2), h, g);  // sqrt(e2)
    r = 2.0 * h;
    r = fma(fma(-g, r, 1.0), r, r);
    double q = tol * r;
    q = fma(fma(-g, q, tol), r, q);  // tol / sqrt(e2)
    constexpr double kInv = 1.0 / 11.09;
    const double w = q * kInv;
    return fma(fma(-11.09, w, q), kInv, w);
}
FQSL_COLD double scale_argument_wide(double tol, double e2) { return tol / sqrt(e2) / 11.09; }

FQSL_COLD double fifth_root(double q) { return pow(q, 0.2); }

// A step and whether the attempt was accepted.
struct Step {
    double s;
    bool accepted;
};
FQSL_HD Step step_of_scale(double s, double scale) {
    if (scale < 0.618) return Step{s * 0.618, false};
    s = s * scale;
    if (s > 100.) s = 100.;
    if (s < 1. / 10.) s = 1. / 10.;
    return Step{s, true};
}
// Where the estimates hold: nothing under- or overflows, in double nor in the float of
// q (below 1e35), and a step beyond its upper bound was not rejected.  Zero, infinite, NaN
// and extreme values go as written, and so does a trace with a first step s0 of 160 or
// more (later ones are at most 100 or smaller than it): `limit` is step_tol_limit(s0).
FQSL_HD double step_tol_limit(double s0) { return s0 < 160.0 ? 1e6 : 0.0; }
FQSL_HD bool step_is_plain(double tol, double e2, double limit) {
    return e2 > 1e-60 && e2 < 1e60 && tol > 1e-60 && tol < limit;
}

// The step after an attempt with step s, from q = tol / err / 11.09 and g, which is q^0.2
// within 1e-5, or NaN.  The library's pow, most of the controller, runs only where its
// value counts: not where g already tells that the step is rejected or that the new one
// lies beyond its bounds.
FQSL_HD Step step_of_argument(double s, double q, float g) {
    double scale = (double)g;
    const double far = s * scale;
    if (!(g < 0.617f || far > 100.1 || (g > 0.619f && far < 0.0999))) scale = fifth_root(q);
    return step_of_scale(s, scale);
}

}  // namespace fqsl
