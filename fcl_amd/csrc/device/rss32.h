// FP32 interval around the RSS distance of a BVTT node (distance(R0, T0, RSS,
// RSS), math/bv/RSS-inl.h:1956-1974: rectangle distance minus both radii,
// clamped at 0): the FP64 value lies in [lo, hi].
//
// The rectangles
//   A = {s e0 + t e1 : 0 <= s <= a0, 0 <= t <= a1}          (A's frame)
//   B = {Tab + Rab (u e0 + v e1) : 0 <= u <= b0, 0 <= v <= b1}
// have a point p of A and a point q of B near their closest ones from
// kRounds alternating projections (14 instructions each, no branch; the FP64
// form's case analysis runs up to 16 edge pairs).  hi is |p - q| minus the
// radii: both points are in their rectangles.  lo is weak duality along
// p to q: for any direction d with |d| <= 1 the rectangles are at least
//   gap(d) = d.Tab + min(0, b0 d.Rab_c0) + min(0, b1 d.Rab_c1)
//            - max(0, a0 d0) - max(0, a1 d1)
// apart (min over B of d.x minus max over A of d.x), with equality for the
// direction of the closest points.  So neither end trusts that the iteration
// has converged; a poor pair only widens the interval.  Over the traversals of
// 20,480-triangle meshes two or more rounds leave 0.26 % of the decisions
// between two children open, as 16 do.
//
// Both ends give way by a rounding margin
//   M = KS*u32*S_T + KR*u32*(a0+a1+b0+b1) + 4*u32*(r1+r2) + 4e-7,  u32 = 2^-24
// (the last since the reference's edge tests compare with an absolute 1e-7,
// RSS-inl.h:485-509, which its value can be off by in small models), with
// S_T = |c1|_1 + |T0|_1 + |c2|_1 (c: the RSS origins).  Derivation (first
// order, fmaf chains with error <= gamma_3 of their terms): Rab and Tab are
// formed as in the OBB cull (cull32.h), each Rab entry within 13u of
// the exact product of the FP64 inputs and each Tab entry within 16.5u S_T;
// so d.Tab errs by <= sqrt(3)*16.5u S_T + 3u*sqrt(3) S_T (its own rounding),
// each b d.Rab_c term by <= (sqrt(3)*13 + 3*sqrt(3) + 2)u b, each a d term
// by <= 2u a, the four additions by <= 4u (S_T + a0+a1+b0+b1), and the
// radius subtraction by <= 2u (|gap| + r1 + r2 + M).  That is < 42u S_T +
// 36u (b0+b1) + 8u (a0+a1) + 3u (r1+r2), and |p - q| errs by less: its three
// coordinates by 16.5u S_T + 16u (b0+b1) + 2u (a0+a1) + 3u of their size,
// and its square root by the factor that hi is raised by.  KS = 72 and KR =
// 60 also cover the second-order terms, the FP64 rounding of the reference's
// own bound and of the RSS fit (~1e-15 relative), and a relative rotation
// whose columns are orthonormal to rss_rotation()'s tolerance.
//
// lo never exceeds the exact distance between the stored FP64 volumes, hence
// never the distance of any triangle pair they contain: a subtree whose lo is
// above the best distance found holds no pair that could be reported.
#pragma once
#include <hip/hip_runtime.h>

#include "cull32.h"
#include "dist64.h"

namespace fclx {

constexpr float kRssKS = 72.0f;
constexpr float kRssKR = 60.0f;
constexpr float kRssAbs = 4e-7f;
constexpr int kRssRounds = 3;

// The FP64 bound takes R's inverse to be its transpose; the margin covers
// what that can differ from here.
__device__ __forceinline__ bool rss_rotation(const M3& R) {
  bool ok = true;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = i; j < 3; ++j) {
      const double g = dot(row(R, i), row(R, j)) - (i == j ? 1.0 : 0.0);
      ok = ok && fabs(g) < 4e-7;
    }
  return ok;
}

// KS*u32*(rcmax1 + |T0|_1 + rcmax2) for a query, rounded up to float;
// infinite (every interval is open) where R0 is no rotation.
__device__ __forceinline__ float rss_margin32(double rcmax1, double rcmax2, const M3& R0,
                                              const V3& T0) {
  if (!rss_rotation(R0)) return INFINITY;
  const double st = (rcmax1 + rcmax2) + ((fabs(T0.x) + fabs(T0.y)) + fabs(T0.z));
  return static_cast<float>(st * (static_cast<double>(kRssKS) * 5.9604644775390625e-08) *
                            (1.0 + 1e-6));
}

__device__ __forceinline__ float clamp32(float x, float top) { return fminf(fmaxf(x, 0.0f), top); }

// [lo, hi] of the RSS distance of (n1, n2) under the query's relative pose R0
// (9, row-major), T0 (3) in float, ms = rss_margin32(...).  hi <= 0: the FP64
// distance is exactly 0.  (NaN inputs give lo = 0 and no finite hi.)
__device__ __forceinline__ void rss_interval32(const float* R0, const float* T0, float ms,
                                               const RssNode32& n1, const RssNode32& n2, float& lo,
                                               float& hi) {
  const float* A1 = n1.axis;
  const float* A2 = n2.axis;
  float P[6], Tt[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      P[3 * j + i] = fdot3(R0[3 * i], R0[3 * i + 1], R0[3 * i + 2], A2[j], A2[3 + j], A2[6 + j]);
    Tt[i] = (fdot3(R0[3 * i], R0[3 * i + 1], R0[3 * i + 2], n2.to[0], n2.to[1], n2.to[2]) +
             T0[i]) -
            n1.to[i];
  }
  float B0[3], B1[3], T[3];  // Rab's first two columns, Tab
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    B0[i] = fdot3(A1[i], A1[3 + i], A1[6 + i], P[0], P[1], P[2]);
    B1[i] = fdot3(A1[i], A1[3 + i], A1[6 + i], P[3], P[4], P[5]);
    T[i] = fdot3(A1[i], A1[3 + i], A1[6 + i], Tt[0], Tt[1], Tt[2]);
  }
  const float a0 = n1.l[0], a1 = n1.l[1], b0 = n2.l[0], b1 = n2.l[1];
  const float c0 = -fdot3(B0[0], B0[1], B0[2], T[0], T[1], T[2]);
  const float c1 = -fdot3(B1[0], B1[1], B1[2], T[0], T[1], T[2]);
  float u = 0.5f * b0, v = 0.5f * b1;
  float s = clamp32(fmaf(u, B0[0], fmaf(v, B1[0], T[0])), a0);
  float t = clamp32(fmaf(u, B0[1], fmaf(v, B1[1], T[1])), a1);
#pragma unroll
  for (int k = 0; k < kRssRounds; ++k) {
    u = clamp32(fmaf(s, B0[0], fmaf(t, B0[1], c0)), b0);
    v = clamp32(fmaf(s, B1[0], fmaf(t, B1[1], c1)), b1);
    s = clamp32(fmaf(u, B0[0], fmaf(v, B1[0], T[0])), a0);
    t = clamp32(fmaf(u, B0[1], fmaf(v, B1[1], T[1])), a1);
  }
  const float d0 = fmaf(u, B0[0], fmaf(v, B1[0], T[0])) - s;
  const float d1 = fmaf(u, B0[1], fmaf(v, B1[1], T[1])) - t;
  const float d2 = fmaf(u, B0[2], fmaf(v, B1[2], T[2]));
  const float nn = fdot3(d0, d1, d2, d0, d1, d2);
  const float rr = n1.r + n2.r;
  const float M = (ms + kRssAbs) + kCullU * (kRssKR * ((a0 + a1) + (b0 + b1)) + 4.0f * rr);
  const bool sized = nn < 1e30f;  // not NaN, no overflow
  const float len = sqrtf(fmaxf(nn, 1e-30f));
  hi = sized ? (len * 1.000002f - rr) + M : INFINITY;
  // |d| <= 1 with room for the rounding of sqrt, the division and the products
  const float sc = 0.999998f / len;
  const float e0 = d0 * sc, e1 = d1 * sc, e2 = d2 * sc;
  const float p0 = fdot3(e0, e1, e2, B0[0], B0[1], B0[2]);
  const float p1 = fdot3(e0, e1, e2, B1[0], B1[1], B1[2]);
  const float gap = (((fdot3(e0, e1, e2, T[0], T[1], T[2]) + fminf(0.0f, b0 * p0)) +
                      fminf(0.0f, b1 * p1)) -
                     fmaxf(0.0f, a0 * e0)) -
                    fmaxf(0.0f, a1 * e1);
  const float l = (gap - rr) - M;
  // touching points have no direction, which proves nothing
  lo = sized && nn > 1e-30f && l > 0.0f ? l : 0.0f;  // (NaN gives 0)
}

}  // namespace fclx
