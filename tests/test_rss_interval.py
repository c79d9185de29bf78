"""The FP32 interval around the RSS distance (device/rss32.h), compiled for the
host: it holds the FP64 bound for random, parallel, touching, far and
degenerate rectangles (zero lengths and radii) at several scales, is open
where the relative pose is no rotation or a number is not finite, and is
narrow enough to decide nearly all of them."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cmath>
#include <cstdint>
#define __device__
#define __forceinline__ inline
using std::fabs; using std::isnan; using std::sqrt;
"""

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include <random>
#include "device/rss32.h"
using namespace fclx;
static std::mt19937_64 g(7);
static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(g); }
static int pick(int n) { return static_cast<int>(g() % n); }
static void rotation(double* R) {
  double q[4], s = 0;
  for (double& x : q) { x = std::normal_distribution<double>()(g); s += x * x; }
  s = std::sqrt(s);
  const double w = q[0] / s, x = q[1] / s, y = q[2] / s, z = q[3] / s;
  const double M[9] = {1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                       2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                       2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)};
  for (int i = 0; i < 9; ++i) R[i] = M[i];
}
static void node(RssNode64& n, RssNode32& f, double scale, int form) {
  rotation(n.axis);
  if (form & 1) for (int i = 0; i < 9; ++i) n.axis[i] = i % 4 == 0;  // axes shared: parallel
  for (double& t : n.to) t = uni(-1, 1) * scale;
  if (form & 1) n.to[2] = std::floor(n.to[2] / scale * 4) * scale / 4;  // coplanar at times
  for (double& l : n.l) l = pick(5) ? std::exp(uni(-7, 0)) * scale : 0.0;
  n.r = pick(4) ? std::exp(uni(-9, -1)) * scale : 0.0;
  for (int i = 0; i < 9; ++i) f.axis[i] = static_cast<float>(n.axis[i]);
  for (int i = 0; i < 3; ++i) f.to[i] = static_cast<float>(n.to[i]);
  for (int i = 0; i < 2; ++i) f.l[i] = static_cast<float>(n.l[i]);
  f.r = static_cast<float>(n.r);
}
int main(int, char** argv) {
  const double scale = std::atof(argv[1]);
  long wide = 0, zero = 0;
  const int total = 400000;
  for (int k = 0; k < total; ++k) {
    const int form = pick(4);
    RssNode64 a, b;
    RssNode32 af, bf;
    node(a, af, scale, form);
    node(b, bf, scale, form);
    M3 R;
    rotation(R.m);
    if (form & 1) for (int i = 0; i < 9; ++i) R.m[i] = i % 4 == 0;
    const double far = pick(8) ? 1 : 1000;
    V3 T = v3(uni(-1, 1) * scale * far, uni(-1, 1) * scale * far, form & 1 ? 0.0 : uni(-1, 1) * scale);
    if (pick(50) == 0) { b = a; bf = af; T = v3(0, 0, 0); }
    double rc[2] = {0, 0};
    for (int i = 0; i < 3; ++i) { rc[0] += std::fabs(a.to[i]); rc[1] += std::fabs(b.to[i]); }
    const int spoil = pick(64);  // what no interval may be closed around
    if (spoil == 0) R.m[pick(9)] += 0.01;
    if (spoil == 1) T.y = NAN;
    if (spoil == 2) af.l[0] = NAN;
    if (spoil == 3) T.x = 1e200;
    float R0[9], T0[3] = {static_cast<float>(T.x), static_cast<float>(T.y), static_cast<float>(T.z)};
    for (int i = 0; i < 9; ++i) R0[i] = static_cast<float>(R.m[i]);
    float lo, hi;
    rss_interval32(R0, T0, rss_margin32(rc[0], rc[1], R, T), af, bf, lo, hi);
    if (spoil < 4) {
      if (lo != 0 || hi < 1e30f) { std::printf("closed %d: %g %g\n", spoil, lo, hi); return 1; }
      continue;
    }
    const double d = rss_distance64(R, T, a, b);
    if (!(lo >= 0) || lo > d || (hi <= 0 ? d != 0 : d > hi)) {
      std::printf("case %d form %d: %.17g not in [%.9g, %.9g]\n", k, form, d, lo, hi);
      return 1;
    }
    zero += d == 0;
    wide += hi - lo > 1e-3 * scale * far && hi > 0;
  }
  std::printf("wide %ld zero %ld of %d\n", wide, zero, total);
  return wide > total / 20 || zero < total / 200;
}
"""


@pytest.mark.parametrize("scale", ["1", "1e-3", "1e4"])
def test_interval_holds_the_fp64_bound(tmp_path, scale):
    d = tmp_path
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(d), "-I",
                    os.path.join(REPO, "fcl_amd", "csrc"), str(d / "main.cpp"), "-o", str(d / "t")],
                   check=True)
    r = subprocess.run([str(d / "t"), scale], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
