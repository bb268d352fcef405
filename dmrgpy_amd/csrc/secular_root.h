// One root of the secular equation of a rank-one update,
//   f(x) = 1/rho + sum_i z_i^2 / (d_i - x) = 0   (poles d ascending, rho > 0),
// for the divide and conquer (tridiag_dc.hip).  Plain arithmetic around a
// callable that sums over the poles, shared by the kernel and the host, so a
// host program can check its convergence without a GPU.
#pragma once

#include <cmath>

#ifdef __HIPCC__
#define DMRG_SECULAR_FN __host__ __device__ __forceinline__
#else
#define DMRG_SECULAR_FN inline
#endif

namespace dmrg {

struct SecularSums {   // of the poles up to j (psi <= 0) and past j (phi >= 0), and their derivatives
  double psi, dpsi, phi, dphi;
};

struct SecularRoot {
  double tau;        // root - origin
  double residual;   // |f| relative to the sum of the terms' sizes
  int next;          // origin: 0 pole j, 1 pole j + 1
  int steps;
};

constexpr int SECULAR_STEPS = 50;

// Root j, between poles dj and dn = d_{j+1} (with weights zj, zn), or past the
// last pole dj (end; z2 = sum of all z_i^2), as the distance tau from the
// nearer pole, so that every difference d_i - x is formed without
// cancellation.  sums(origin, tau) evaluates at x = origin + tau.
//
// Two-pole rational steps with the nearer pole's weight exact (the fixed
// weight method of Li, LAPACK Working Note 89); the last root has one pole
// with the slope of all.  A root much closer to its pole than the start can
// make them creep (halving tau, or lost in the rounding of tau + step), so a
// step that leaves the bracket or follows one that left more than a quarter
// of |f| is replaced by the geometric mean of the bracket, whose ends both
// have the sign of tau: the term of the nearer pole alone bounds |tau| from
// below.  Weights down to 1e-35 and gaps down to 1e-60 of the largest take at
// most 18 evaluations; steps from the weights of the middle way with
// arithmetic bisection, used before, ran out of 50.
template <class Sums>
DMRG_SECULAR_FN SecularRoot secular_root(bool end, double dj, double dn, double zj, double zn, double z2, double rinv,
                                         Sums sums) {
  constexpr double eps = 1.1102230246251565e-16;   // 2^-53
  SecularRoot r;
  r.next = 0;
  const double gap = dn - dj;   // unused at the end
  double origin = dj, lo, hi, tau = 0.5 * (end ? z2 / rinv : gap);
  SecularSums s = sums(origin, tau);
  double f = rinv + s.psi + s.phi;
  if (end) {
    lo = zj * zj / rinv * (1.0 - 16.0 * eps);
    hi = z2 / rinv * (1.0 + 16.0 * eps);
  } else if (f < 0.0) {   // nearer the right pole
    r.next = 1;
    origin = dn;
    lo = -tau;
    hi = -fmin(tau, zn * zn / fabs(s.psi)) * (1.0 - 1e-10);
    tau = -tau;
  } else {
    lo = fmin(tau, zj * zj / (rinv + s.phi)) * (1.0 - 1e-10);
    hi = tau;
  }
  bool slow = false;
  int it = 0;
  for (; it < SECULAR_STEPS; ++it) {
    if (!(fabs(f) > 8.0 * eps * (rinv + fabs(s.psi) + fabs(s.phi)))) break;
    if (f < 0.0) lo = fmax(lo, tau);
    else hi = fmin(hi, tau);
    const double ej = (dj - origin) - tau, df = s.dpsi + s.dphi;
    double x;
    if (end) {
      const double c = f - s.dpsi * ej;
      x = tau + ej + s.dpsi * ej * ej / c;
    } else {
      const double en = (dn - origin) - tau;
      const double q = r.next ? zn / en : zj / ej;
      const double c = r.next ? f - ej * df - gap * q * q : f - en * df + gap * q * q;
      const double a = (ej + en) * f - ej * en * df, b = ej * en * f;
      const double disc = sqrt(fabs(a * a - 4.0 * b * c));
      x = tau + (a <= 0.0 ? (a - disc) / (2.0 * c) : 2.0 * b / (a + disc));
    }
    const bool mean = slow || !(x > lo && x < hi);
    if (mean) {
      const double p = fmin(fabs(lo), fabs(hi)), q = fmax(fabs(lo), fabs(hi));
      x = q > 2.0 * p ? copysign(sqrt(p) * sqrt(q), tau) : 0.5 * (lo + hi);
    }
    if (x == tau) break;
    tau = x;
    const double before = f;
    s = sums(origin, tau);
    f = rinv + s.psi + s.phi;
    slow = !mean && fabs(f) > 0.25 * fabs(before);
  }
  r.tau = tau;
  r.residual = fabs(f) / (rinv + fabs(s.psi) + fabs(s.phi));
  r.steps = it;
  return r;
}

}  // namespace dmrg
