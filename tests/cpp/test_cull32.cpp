// The FP32 cull against the FP64 test it stands for, on the host: node pairs
// whose sizes run over the range of a double, at every distance from far apart
// to one inside the other.  argv[1]: pairs per scale.  Prints, per scale, the
// sure verdicts, the unsure ones and the wrong ones.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../fcl_amd/csrc/device/query32.h"

using namespace fclx;

namespace {

std::mt19937_64 rng(7);
double uniform(double lo, double hi) {
  return std::uniform_real_distribution<double>(lo, hi)(rng);
}

void rotation(double* R) {
  double q[4], n = 0;
  for (double& x : q) {
    x = std::normal_distribution<double>()(rng);
    n += x * x;
  }
  n = std::sqrt(n);
  const double w = q[0] / n, x = q[1] / n, y = q[2] / n, z = q[3] / n;
  const double m[9] = {1 - 2 * (y * y + z * z), 2 * (x * y - w * z),     2 * (x * z + w * y),
                       2 * (x * y + w * z),     1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                       2 * (x * z - w * y),     2 * (y * z + w * x),     1 - 2 * (x * x + y * y)};
  for (int k = 0; k < 9; ++k) R[k] = m[k];
}

// A node of size s, a cube or a sliver, around a centre up to `far` sizes away.
void node(double s, double far, bool cube, ObbNode64& n, ObbNode32& f) {
  rotation(n.axis);
  for (int k = 0; k < 3; ++k) {
    n.to[k] = s * far * uniform(-1, 1);
    n.extent[k] = s * (cube ? uniform(0.8, 1) : std::exp(uniform(-4, 0)));
  }
  n.first_child = f.first_child = 0;
  n.pad = 0;
  for (int k = 0; k < 9; ++k) f.axis[k] = static_cast<float>(n.axis[k]);
  for (int k = 0; k < 3; ++k) {
    f.to[k] = static_cast<float>(n.to[k]);
    f.extent[k] = static_cast<float>(n.extent[k]);
  }
}

double norm1(const double* v) { return std::fabs(v[0]) + std::fabs(v[1]) + std::fabs(v[2]); }

}  // namespace

int main(int argc, char** argv) {
  const int pairs = argc > 1 ? std::atoi(argv[1]) : 1000;
  // in steps of a tenth where floats end
  for (double e = -320; e < 306.5; e += e < -50 || e > 45 ? 10 : (e > 36.9 && e < 41 ? 0.1 : 1)) {
    long sure = 0, unsure = 0, wrong = 0;
    for (int i = 0; i < pairs; ++i) {
      // the second node's size and place relative to the first's
      const bool cube = i % 4 == 0;
      const double s = std::pow(10.0, e) * (cube ? 1 : uniform(1, 10));
      const double other = cube ? s : s * std::exp(uniform(-3, 3)), far = i % 3 == 0 ? 8.0 : 0.7;
      ObbNode64 a, b;
      ObbNode32 fa, fb;
      node(s, far, cube, a, fa);
      node(other, far, cube, b, fb);
      double R[9], T[3];
      rotation(R);
      for (double& t : T) t = (s + other) * uniform(-1, 1) * (i % 2 ? 1.2 : 0.1);
      if (i % 7 == 0) {  // far from the origin, but next to each other
        for (int k = 0; k < 3; ++k) {
          const double away = 30 * s * uniform(-1, 1);
          a.to[k] += away;
          T[k] += away;
          fa.to[k] = static_cast<float>(a.to[k]);
        }
      }
      QueryXf32 X;
      make_xf32(R, T, norm1(a.to), norm1(b.to), X);
      M3 R0;
      for (int k = 0; k < 9; ++k) R0.m[k] = R[k];
      const int got = obb_cull32(X, fa, fb);
      const int want = obb_overlap64(R0, v3(T[0], T[1], T[2]), a, b) ? kCullOverlap : kCullDisjoint;
      if (got == kCullUnsure)
        ++unsure;
      else if (got == want)
        ++sure;
      else
        ++wrong;
    }
    std::printf("%.1f %ld %ld %ld\n", e, sure, unsure, wrong);
  }
  return 0;
}
