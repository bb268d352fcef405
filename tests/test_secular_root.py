"""The divide and conquer's root finder (dmrgpy_amd/csrc/secular_root.h),
compiled for the host with g++ and run on secular equations that deflation
leaves over (CPU): weights down to 1e-35, gaps down to 1e-60 of the largest,
couplings from 1e-20 to 2, among them the two that made rational steps creep --
a weight so small that the root lies within the rounding of one step, and the
other terms vanishing at the pole itself.

Every root is found in fewer steps than the limit (30 of 50 are asserted) with
a residual of rounding size: |f| in long double against the sum of the terms'
sizes within (40 + K) 2^-53, the summation error of K terms plus the stopping
rule's 8 2^-53 and the rounding of tau (one ulp moves a term by its own size
times 2^-53).
"""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, os.pardir, "dmrgpy_amd", "csrc")

HARNESS = r"""
#include "secular_root.h"
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>
using namespace dmrg;
typedef std::vector<double> vec;
static const double EPS = 1.1102230246251565e-16;

// what deflation would leave: weights the update sees, poles far enough apart
static void deflate(vec& d, vec& z, double rho) {
  double mx = 0.0;
  for (double x : d) mx = std::max(mx, std::fabs(x));
  vec dd, zz;
  for (size_t i = 0; i < d.size(); ++i) {
    if (!(rho * std::fabs(z[i]) > std::max(EPS * std::fabs(d[i]), 1e-40 * mx))) continue;
    if (!dd.empty()) {
      const double p = dd.back(), zp = zz.back();
      if (std::fabs((d[i] - p) * zp * z[i]) <= EPS * (std::fabs(p) + std::fabs(d[i])) * (zp * zp + z[i] * z[i])) {
        zz.back() = std::hypot(zp, z[i]);
        continue;
      }
    }
    dd.push_back(d[i]);
    zz.push_back(z[i]);
  }
  d = dd;
  z = zz;
}

static int max_steps;
static double max_res;
static long long roots;

static void solve(vec d, vec z, double rho) {
  deflate(d, z, rho);
  const int K = (int)d.size();
  double z2 = 0.0;
  for (double x : z) z2 += x * x;
  for (int j = 0; j < K; ++j) {
    const bool end = j == K - 1;
    const int jn = end ? j : j + 1;
    const double rinv = 1.0 / rho;
    const SecularRoot r = secular_root(end, d[j], d[jn], z[j], z[jn], z2, rinv, [&](double origin, double tau) {
      SecularSums s = {0.0, 0.0, 0.0, 0.0};
      for (int i = 0; i < K; ++i) {
        const double t = z[i] / ((d[i] - origin) - tau);
        (i <= j ? s.psi : s.phi) += z[i] * t;
        (i <= j ? s.dpsi : s.dphi) += t * t;
      }
      return s;
    });
    const double origin = r.next ? d[j + 1] : d[j];
    long double f = (long double)rinv, size = (long double)rinv;
    for (int i = 0; i < K; ++i) {
      const long double t = (long double)z[i] * z[i] / (((long double)d[i] - origin) - r.tau);
      f += t;
      size += std::fabs(t);
    }
    const bool inside = r.next ? r.tau < 0.0 : r.tau > 0.0;
    const double res = inside ? (double)(std::fabs(f) / size) / (EPS * (40 + K)) : 1e300;
    max_steps = std::max(max_steps, r.steps);
    if (!(res <= max_res)) max_res = res;
    ++roots;
  }
}

int main() {
  std::mt19937_64 gen(7);
  auto u = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(gen); };
  std::normal_distribution<double> g;
  const char* names[] = {"random", "gaps", "weights", "graded", "clusters", "at the pole"};
  for (int kind = 0; kind < 6; ++kind) {
    max_steps = 0;
    max_res = 0.0;
    roots = 0;
    for (int t = 0; t < 400; ++t) {
      const int K = kind == 5 ? 3 : 1 + (int)(gen() % 60);
      vec d(K), z(K);
      double at = 0.0;
      for (int i = 0; i < K; ++i) {
        d[i] = g(gen);
        z[i] = g(gen);
        if (kind == 1) { d[i] = at += std::pow(10.0, u(-15, 0)); z[i] = std::pow(10.0, u(-30, 0)); }
        if (kind == 2) z[i] = std::pow(10.0, u(-20, 0));
        if (kind == 3) { d[i] = std::pow(10.0, u(-60, 0)); z[i] = std::pow(10.0, u(-35, 0)); }
        if (kind == 4) { d[i] = std::round(100 * d[i]) / 100 + 1e-9 * g(gen); z[i] *= std::pow(10.0, u(-8, 0)); }
      }
      std::sort(d.begin(), d.end());
      double rho = kind == 0 ? u(0.01, 2.0) : std::pow(10.0, u(-20, 0.3));
      if (kind == 5) {   // 1/rho + z0^2 / (d0 - d1) + z2^2 / (d2 - d1) = 0 to rounding
        d = {0.0, u(0.2, 0.8), 2.0};
        z = {u(0.3, 0.9), std::pow(10.0, u(-20, -2)), u(0.1, 0.3)};
        rho = 1.0 / (z[0] * z[0] / d[1] - z[2] * z[2] / (d[2] - d[1]));
        if (!(rho > 0.0)) continue;
      } else {
        double n = 0.0;
        for (double x : z) n += x * x;
        for (double& x : z) x /= std::sqrt(n);
      }
      solve(d, z, rho);
    }
    std::printf("%s;%lld;%d;%.3g\n", names[kind], roots, max_steps, max_res);
  }
  return 0;
}
"""


def test_roots_are_found(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "harness.cpp", tmp_path / "harness"
    src.write_text(HARNESS)
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    lines = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")
    rows = [line.split(";") for line in lines if line]
    assert len(rows) == 6
    for name, roots, steps, res in rows:
        print(name, "roots", roots, "steps", steps, "residual / bound", res)
        assert int(roots) > 200, name
        assert int(steps) < 30, (name, steps)
        assert float(res) <= 1.0, (name, res)
