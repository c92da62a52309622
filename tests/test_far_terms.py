"""The rounding bound of the far-from-equilibrium root-find's FP32 polynomial
(csrc/far_terms.h), compiled for the host: over random nodes whose x = D / f
reach 0.02 to 1.5, at centres a and steps d within the trust radius, the
polynomial's error against sums in extended precision stays within the stated
slack, and z is rounded once.  Nodes with all D of one kind (each term rounded the same way, nothing
cancels) come nearest to it."""
import os
import subprocess

from conftest import PKG_DIR

SOURCE = r"""
#include <cmath>
#include <cstdio>
#include <random>
#include "far_terms.h"
#ifndef TERMS
#define TERMS uclbs::FarTerms<6>
#endif
int main() {
  std::mt19937_64 r(5);
  std::uniform_real_distribution<double> u(-1, 1);
  double worst = 0.0, zworst = 0.0, rounding = 0.0;
  for (int trial = 0; trial < 200000; ++trial) {
    const double x = std::pow(10.0, -2 + 2 * std::fabs(u(r))), a = 2.0 + 0.3 * u(r);
    TERMS w;
    w.clear();
    w.add(1.0f, x, 1.0 / (1.0 + a * x));
    const long double z = (long double)x / (1.0L + (long double)a * x);
    rounding = std::fmax(rounding, (double)std::fabs(w.zmax / z - 1));
  }
  for (int trial = 0; trial < 600000; ++trial) {
    const double size = std::pow(10.0, -0.75 + 0.95 * u(r)), a = 2.0 + 0.3 * u(r);
    // mixed signs; positive; one x; few large; one x and f (27 equal roundings)
    const int kind = trial % 5;
    const double one = 0.5 + 0.5 * std::fabs(u(r)), same = 0.02 + 0.1 * std::fabs(u(r));
    TERMS w;
    w.clear();
    long double T[7] = {};
    double zmax = 0.0;
    for (int i = 0; i < 27; ++i) {
      const double f = kind == 4 ? same : 0.02 + 0.1 * std::fabs(u(r));
      double x = size * (kind == 2 || kind == 4 ? one : kind == 3 && i % 9 ? 1e-3 * u(r) : u(r));
      if (kind == 1) x = std::fabs(x);
      const float D = (float)(f * x);
      x = D / f;
      const double A = 1.0 + a * x;
      if (A <= 0.02) continue;
      w.add(D, x, 1.0 / A);
      const long double z = (long double)x / (1.0L + (long double)a * x);
      zmax = std::fmax(zmax, std::fabs((double)z));
      long double t = D;
      for (int n = 2; n <= 6; ++n) T[n] += (t *= z);
    }
    zworst = std::fmax(zworst, zmax / w.zbound());
    for (int k = 1; k <= 4; ++k) {
      const double d = (k & 1 ? 1 : -1) * 0.5 / zmax * std::pow(10.0, 1 - k);
      long double e = 0.0L, dn = d;
      for (int n = 2; n <= 6; ++n) {
        dn *= d;
        e += (n & 1 ? -1 : 1) * ((long double)w.T[n] - T[n]) * dn / (n * (n - 1));
      }
      worst = std::fmax(worst, (double)std::fabs(e) / w.slack(d));
    }
  }
  printf("%.6f %.9f %.3e\n", worst, zworst, rounding);
}
"""


def measured(tmp_path, flags=()):
    (tmp_path / "terms.cpp").write_text(SOURCE)
    exe = str(tmp_path / "terms")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wno-unknown-pragmas", "-D__host__=", "-D__device__=",
                    "-D__forceinline__=inline", *flags, "-I", os.path.join(PKG_DIR, "csrc"),
                    str(tmp_path / "terms.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return [float(v) for v in out.split()]


def test_slack_covers_the_rounding(tmp_path):
    worst, z, rounding = measured(tmp_path)
    print(f"largest error over slack {worst:.3f}, max |z| over its bound {z:.9f}, z {rounding:.2e}")
    assert rounding <= 1.001 * 2.0 ** -24  # z is a rounded FP64 value
    assert worst <= 1.0 and z <= 1.0
    assert worst > 0.05  # the bound is of the size of what it bounds
