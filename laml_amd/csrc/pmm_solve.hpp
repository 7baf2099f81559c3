// The scalar solves of the M-step: branch lengths and nu (EM_solver.py:328-407).
// Plain arithmetic on doubles, so that the same source also compiles for the
// host, with an estimate of the reciprocal in place of
// __builtin_amdgcn_rcp.
#pragma once
#include <math.h>

namespace laml {

// 1 / x where x and 1 / x are normal numbers: the hardware estimate and two
// Newton steps (no scaling for extreme arguments)
__device__ __forceinline__ double rcp_normal(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// 1 / expm1(y) for y > 0.  Past 700 the quotient is below 1e-304, which no sum
// of the solves resolves, and from 709.8 on expm1 is infinite, of which the
// Newton steps of rcp_normal would make inf * 0: the value at 700 there.
// (fmin drops a NaN; every caller has one beside it then, from a count, a
// length or nu itself.  A comparison and a selection in its place cost an EM
// step of 250 x 30 3 %.)
__device__ __forceinline__ double rcp_expm1(double y) { return rcp_normal(expm1(fmin(y, 700.0))); }

constexpr double kEpsNu = 1e-5;   // EM_solver.py:307 eps_nu
constexpr double kEpsS = 1e-6;    // EM_solver.py:307 eps_s

// The branch and nu solves look for the root of a decreasing function g of
// x > 0 that behaves like S/x - A for small x, through G(x) = x g(x), which is
// nearly linear.  From g and its first three derivatives at x: the root of G's
// cubic Taylor polynomial, as a step from x (a plain Newton step where the
// polynomial gives none near).  The step's own error is of the fourth order:
// one of at most kBranchDone x or kNuDone x ends a solve.  Over two million
// random branch objectives the roots are then within 4.7e-16 of the true ones
// in the default box and 2.3e-15 in [1e-6, 1000], Newton steps to 1e-13 x
// within 4.7e-16 and 4.7e-14 (ending at 1e-4 x: 1.9e-15 and 1.3e-14); over
// 20,000 nu problems within 3.3e-16, Newton steps to 1e-12 x within 3.6e-16.  A
// warm-started solve takes one or two evaluations where Newton steps took four
// to seven.
constexpr double kBranchDone = 6e-5;
constexpr double kNuDone = 1e-4;
__device__ __forceinline__ double taylor_step(double x, double g, double g1, double g2, double g3) {
  const double c0 = x * g, c1 = fma(x, g1, g), c2 = fma(0.5 * x, g2, g1), c3 = fma(x * (1.0 / 6.0), g3, 0.5 * g2);
  const double t0 = -c0 / c1;
  double t = t0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const double p = fma(fma(fma(c3, t, c2), t, c1), t, c0);
    const double q = fma(fma(3.0 * c3, t, 2.0 * c2), t, c1);
    t -= p * rcp_normal(q);
  }
  return fabs(t - t0) <= 0.5 * fabs(t0) ? t : t0;
}

struct BranchObj {
  double A, S1, B, nu;  // f'(d) = -A + S1/expm1(d) + B nu/expm1(nu d)
};
// the derivative of the branch objective, g, and its own first three: with
// r = 1 / expm1(y) and s = r (1 + r), r' = -s, s' = -s (1 + 2 r) and
// (s (1 + 2 r))' = -s (1 + 6 s)
struct BranchG {
  double g, g1, g2, g3;
};
__device__ __forceinline__ BranchG branch_g(const BranchObj& o, double d) {
  const double r = rcp_expm1(d);
  const double s = r * (1.0 + r);
  BranchG b;
  b.g = fma(o.S1, r, -o.A);
  b.g1 = -o.S1 * s;
  b.g2 = o.S1 * s * fma(2.0, r, 1.0);
  b.g3 = -o.S1 * s * fma(6.0, s, 1.0);
  if (o.B > 0.0) {
    const double rn = rcp_expm1(o.nu * d);
    const double sn = rn * (1.0 + rn);
    const double B1 = o.B * o.nu, B2 = B1 * o.nu * sn, B3 = B2 * o.nu;
    b.g = fma(B1, rn, b.g);
    b.g1 -= B2;
    b.g2 = fma(B3, fma(2.0, rn, 1.0), b.g2);
    b.g3 = fma(-B3 * o.nu, fma(6.0, sn, 1.0), b.g3);
  }
  return b;
}
// argmax over [dmin, dmax] of the strictly concave branch objective, kept in
// a bracket.  From a start inside the box the bounds are evaluated only when
// a step reaches for them.
__device__ double solve_branch(const BranchObj& o, double dmin, double dmax, double x0) {
  double lo = dmin, hi = dmax;
  bool lo_known = false, hi_known = false;  // whether g(lo) > 0, g(hi) < 0 are known
  double x = x0;
  if (!(x0 > lo && x0 < hi)) {
    if (!(branch_g(o, dmin).g > 0.0)) return dmin;
    if (!(branch_g(o, dmax).g < 0.0)) return dmax;
    lo_known = hi_known = true;
    x = 0.5 * (lo + hi);
  }
  for (int it = 0; it < 100; ++it) {
    const BranchG b = branch_g(o, x);
    if (b.g > 0.0) {
      lo = x;
      lo_known = true;
    } else if (b.g < 0.0) {
      hi = x;
      hi_known = true;
    } else if (b.g == 0.0) {
      return x;
    } else {
      return dmin;  // not a number: as at the lower bound
    }
    const double step = taylor_step(x, b.g, b.g1, b.g2, b.g3);
    double xn = x + step;
    if (fabs(step) <= kBranchDone * x && xn >= dmin && xn <= dmax) return xn;
    if (!(xn > lo && xn < hi)) {
      // out of the bracket: the optimum is at a bound whose slope points out
      if (!lo_known) {
        if (!(branch_g(o, dmin).g > 0.0)) return dmin;
        lo_known = true;
      }
      if (!hi_known) {
        if (!(branch_g(o, dmax).g < 0.0)) return dmax;
        hi_known = true;
      }
      xn = 0.5 * (lo + hi);
    }
    if (hi - lo <= 1e-13 * hi) return xn;
    x = xn;
  }
  return x;
}

// the first evaluation point: the current nu, or 1/2 when outside (0, 1)
__device__ __forceinline__ double nu_start(double nu) { return nu > 0.0 && nu < 1.0 ? nu : 0.5; }

// h'(x) and its first three derivatives
struct NuSum {
  double g, g1, g2, g3;
};

// One bracketed step towards the root of h' from its evaluation at x.
// [lo, hi] brackets the root (hi > 1 until the bound x = 1 has been
// evaluated).  Returns true when the solve has converged; xn is the next
// iterate (the answer when converged).
__device__ __forceinline__ bool nu_step(double x, const NuSum& n, double& lo, double& hi, double& xn) {
  if (n.g > 0.0) lo = x; else if (n.g < 0.0) hi = x;
  if (n.g > 0.0 && x >= 1.0) {
    xn = 1.0;  // optimum at the upper bound
    return true;
  }
  if (n.g == 0.0) {
    xn = x;
    return true;
  }
  const double step = taylor_step(x, n.g, n.g1, n.g2, n.g3);
  const double top = fmin(hi, 1.0);
  xn = x + step;
  if (fabs(step) <= kNuDone * x) {
    xn = fmin(fmax(xn, 0.0), 1.0);
    return true;
  }
  if (xn >= 1.0 && hi > 1.0) xn = 1.0;
  else if (!(xn > lo && xn < top)) xn = 0.5 * (lo + top);
  return top - lo <= 1e-12 * top;
}

// One branch's terms: a = S0 + S1 + S3, b = S2 + S4 of the branch, its length
// dv (derivatives of 1 / expm1 as in branch_g).
__device__ __forceinline__ void nu_term(double a, double bb, double dv, double x, NuSum& n) {
  if (bb == 0.0) return;
  const double r = rcp_expm1(x * dv);
  const double s = r * (1.0 + r);
  const double b2 = bb * dv * dv * s, b3 = b2 * dv;
  n.g = fma(dv, fma(bb, r, -a), n.g);
  n.g1 -= b2;
  n.g2 = fma(b3, fma(2.0, r, 1.0), n.g2);
  n.g3 = fma(-b3 * dv, fma(6.0, s, 1.0), n.g3);
}

}  // namespace laml
