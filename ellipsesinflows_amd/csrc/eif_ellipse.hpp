// eif_ellipse.hpp -- ellipse geometry on the device (src/ellipse.c:7-65): the
// shape's constants, sine and cosine of bounded angles, and the foot of the
// normal by the reference's iteration (foot_fp32 for the start, foot_fp64 to
// its stopping rule).
#pragma once
#include <hip/hip_runtime.h>
#include "eif_internal.hpp"

namespace eif {

// x^3 to nearly correct rounding (error-free square, then product), the
// value glibc's pow(x, 3.) returns.
__device__ inline double cube(double x) {
  const double p = x * x;
  const double e = fma(x, x, -p);
  const double h = p * x;
  const double eh = fma(p, x, -h);
  return h + (eh + e * x);
}

struct EllipseShape {
  double a, b;
  double kex, key;  // a(1-(b/a)^2), b(1-(a/b)^2)   (ellipse.c:7-13)
  double a2b2;      // a*a + b*b                     (ellipse.c:49)
  double ia, ib;    // 1/a, 1/b
};

__device__ inline EllipseShape make_shape(double a, double b) {
  EllipseShape s;
  s.a = a;
  s.b = b;
  const double ba = b / a, ab = a / b;
  s.kex = a * (1. - ba * ba);
  s.key = b * (1. - ab * ab);
  s.a2b2 = a * a + b * b;
  s.ia = 1. / a;
  s.ib = 1. / b;
  return s;
}

struct EllipseShape32 {
  float a, b, kex, key, a2b2;
};

__device__ inline EllipseShape32 shape32(const EllipseShape &e) {
  return {(float)e.a, (float)e.b, (float)e.kex, (float)e.key, (float)e.a2b2};
}

// sin and cos on [0, pi/2] (slightly beyond is fine): Taylor polynomials
// on |u| <= pi/4 (truncation below 1e-20) after u = pi/2 - t for t > pi/4,
// with pi/2 split into two doubles so that the reduction is exact to
// rounding.  The general libm routines carry large-argument reduction
// that is never needed here and costs registers in the cell loop.
__device__ inline double sin_poly(double u) {
  const double u2 = u * u;
  double p = 1. / 355687428096000.;
  p = fma(p, u2, -1. / 1307674368000.);
  p = fma(p, u2, 1. / 6227020800.);
  p = fma(p, u2, -1. / 39916800.);
  p = fma(p, u2, 1. / 362880.);
  p = fma(p, u2, -1. / 5040.);
  p = fma(p, u2, 1. / 120.);
  p = fma(p, u2, -1. / 6.);
  return fma(u * u2, p, u);
}
__device__ inline double cos_poly(double u) {
  const double u2 = u * u;
  double p = -1. / 6402373705728000.;
  p = fma(p, u2, 1. / 20922789888000.);
  p = fma(p, u2, -1. / 87178291200.);
  p = fma(p, u2, 1. / 479001600.);
  p = fma(p, u2, -1. / 3628800.);
  p = fma(p, u2, 1. / 40320.);
  p = fma(p, u2, -1. / 720.);
  p = fma(p, u2, 1. / 24.);
  p = fma(p, u2, -0.5);
  return fma(u2, p, 1.);
}
__device__ inline void sincos_q1(double t, double &s, double &c) {
  constexpr double PIO2_HI = 1.5707963267948966;      // nearest double to pi/2
  constexpr double PIO2_LO = 6.123233995736766e-17;   // pi/2 - PIO2_HI
  // one pair of polynomials for both halves (no divergent branch): the
  // argument and the roles of the results are selected instead
  const bool low = t <= 0.78539816339744831;
  const double u = low ? t : (PIO2_HI - t) + PIO2_LO;
  const double ps = sin_poly(u), pc = cos_poly(u);
  s = low ? ps : pc;
  c = low ? pc : ps;
}

// 1/sqrt(x) from the hardware estimate and one Newton step (relative error
// near 1e-16); used where only the size of a step depends on it
__device__ inline double rsqrt_nr(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.);
  return fma(0.5 * y, e, y);
}

// asin by its Maclaurin series, exact to rounding for |x| <= 2^-6; for
// larger |x| a monotone under-estimate, which only shortens a step of the
// fixed-point iteration (its fixed point is x = 0)
__device__ inline double asin_series(double x) {
  const double x2 = x * x;
  double p = 0.022372159090909091;  // 63/2816
  p = fma(p, x2, 0.030381944444444444);  // 35/1152
  p = fma(p, x2, 0.044642857142857144);  // 5/112
  p = fma(p, x2, 0.075);                 // 3/40
  p = fma(p, x2, 1. / 6.);
  return fma(x * x2, p, x);
}

// cos and sin of t + delta from c = cos t, s = sin t, |delta| <= 2^-10
__device__ inline void rotate_small(double &c, double &s, double delta) {
  const double d2 = delta * delta;
  const double hc = d2 * (0.5 - d2 * (1. / 24.));           // 1 - cos(delta)
  const double sd = delta * (1. - d2 * (1. / 6. - d2 * (1. / 120.)));  // sin(delta)
  const double cn = c - (s * sd + c * hc);
  const double sn = s + (c * sd - s * hc);
  c = cn;
  s = sn;
}

// FP32 part: from t = pi/4 until |dt| < 1e-3 (at most 8 iterations)
__device__ inline float foot_fp32(const EllipseShape32 &f, double px, double py, int &it32) {
  float tf = (float)(0.25 * EIF_PI);
  const float fx = (float)px, fy = (float)py;
  for (int n = 0; n < 8; n++) {
    float sn, cs;
    __sincosf(tf, &sn, &cs);
    const float x = f.a * cs, y = f.b * sn;
    const float ex = f.kex * (cs * cs * cs), ey = f.key * (sn * sn * sn);
    const float rx = x - ex, ry = y - ey;
    const float qx = fx - ex, qy = fy - ey;
    const float rr = rx * rx + ry * ry, qq = qx * qx + qy * qy;
    float arg = (rx * qy - ry * qx) * __builtin_amdgcn_rsqf(rr * qq);
    arg = fminf(fmaxf(arg, -1.f), 1.f);
    const float den = fmaxf(f.a2b2 - x * x - y * y, 1e-30f);
    const float a2 = arg * arg;
    const float as = arg + arg * a2 * (0.16666667f + a2 * (0.075f + a2 * 0.044642857f));
    const float dt = __builtin_amdgcn_sqrtf(rr) * as * __builtin_amdgcn_rsqf(den);
    it32++;
    if (!(fabsf(dt) < 1e30f)) break;  // no usable step: hand over to FP64
    tf = fminf(fmaxf(tf + dt, 0.f), 1.5707963f);
    if (fabsf(dt) < 1e-3f) break;
  }
  return tf;
}

// FP64 part: the reference's iteration and stopping rule from t (updated
// in place); (c, s) = (cos t, sin t) of the foot on the first-quadrant arc
// for the folded point (px, py) >= 0
__device__ inline void foot_fp64(const EllipseShape &e, double px, double py, double &t,
                                 double &c, double &s, int &it64) {
  constexpr double HALF_PI = 0.5 * EIF_PI;
  sincos_q1(t, s, c);
  for (int n = 0;; n++) {
    const double x = e.a * c, y = e.b * s;
    const double ex = e.kex * cube(c), ey = e.key * cube(s);
    const double rx = x - ex, ry = y - ey;
    const double qx = px - ex, qy = py - ey;
    // dt = r asin(cross / (r q)) / sqrt(a^2 + b^2 - x^2 - y^2): the
    // residual (cross) is formed exactly as in ellipse.c:41-46; the scale
    // factors only set the step length, so reciprocal square roots do
    const double rr = ry * ry + rx * rx, qq = qy * qy + qx * qx;
    const double cross = rx * qy - ry * qx;
    const double arg = cross * rsqrt_nr(rr * qq);
    const double dt = asin_series(arg) * (rr * rsqrt_nr(rr * (e.a2b2 - x * x - y * y)));
    double tn = t + dt;
    tn = fmin(HALF_PI, tn);
    tn = fmax(0., tn);
    const double delta = tn - t;
    if (fabs(delta) <= 0x1p-10 && tn != HALF_PI && tn != 0.)
      rotate_small(c, s, delta);
    else
      sincos_q1(tn, s, c);
    t = tn;
    it64++;
    if (fabs(dt) < 1.e-8) break;
    if (n > 100) break;
  }
}

}  // namespace eif
