// Per-query records of the collide engines (FP64 pose with the triangle
// arrays, FP32 pose with the cull margin, node arrays) and the loads and
// descent rule that the FP32-culling traversals share.
#pragma once

#include "cull32.h"
#include "exact64.h"
#include "../fclx_layout.h"

namespace fclx {

// FP64 relative pose of a query plus its meshes' triangle-major vertex
// arrays: everything a triangle test needs, in one 128-B line.
struct alignas(128) QueryXf64 {
  double R[9];
  double T[3];
  const double* tv1;
  const double* tv2;
};

// Node and size arrays of a query's two meshes, read in parallel with the
// query's transform so no mesh-descriptor load sits on the critical path.
struct QueryPtr {
  const ObbNode32* n1;
  const ObbNode32* n2;
  const double* s1;
  const double* s2;
};

// Both ids name live OBBRSS meshes.
__device__ __forceinline__ bool obbrss_query_ok(const MeshDev* meshes, int n, int i1, int i2) {
  if (i1 < 0 || i2 < 0 || i1 >= n || i2 >= n) return false;
  const MeshDev& a = meshes[i1];
  const MeshDev& b = meshes[i2];
  return a.num_bvs > 0 && b.num_bvs > 0 && a.bv_type == 0 && b.bv_type == 0;
}

// R = R1^T R2, T = R1^T (t2 - t1)
__device__ __forceinline__ void rel_pose64(const double* tf1, const double* tf2, double* R,
                                           double* T) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      R[3 * i + j] = (tf1[i] * tf2[j] + tf1[3 + i] * tf2[3 + j]) + tf1[6 + i] * tf2[6 + j];
  const V3 d = v3(tf2[9] - tf1[9], tf2[10] - tf1[10], tf2[11] - tf1[11]);
  T[0] = dot(col(tf1, 0), d);
  T[1] = dot(col(tf1, 1), d);
  T[2] = dot(col(tf1, 2), d);
}

__device__ __forceinline__ void make_xf32(const double* R, const double* T, double cmax1,
                                          double cmax2, QueryXf32& X) {
#pragma unroll
  for (int i = 0; i < 9; ++i) X.R[i] = static_cast<float>(R[i]);
#pragma unroll
  for (int i = 0; i < 3; ++i) X.T[i] = static_cast<float>(T[i]);
  const double st = cmax1 + (fabs(T[0]) + fabs(T[1]) + fabs(T[2])) + cmax2;
  // margin rounded up: the float conversion may round down by <= 2^-24
  X.ms = static_cast<float>((static_cast<double>(kCullKS) * static_cast<double>(kCullU) * st +
                             static_cast<double>(kCullTiny)) *
                            (1.0 + 1.0 / 1048576.0));
}

// The same for a query whose poses may be any matrices: the cull's margin
// holds for rotations, with any other matrix every test is left to FP64.
__device__ __forceinline__ void make_xf32_checked(const double* R, const double* T, double cmax1,
                                                  double cmax2, QueryXf32& X) {
  make_xf32(R, T, cmax1, cmax2, X);
  int unit = 1;  // (without branches)
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    unit &= static_cast<int>(sq(col(R, k)) < 1.0001);
    unit &= static_cast<int>(sq(v3(R[3 * k], R[3 * k + 1], R[3 * k + 2])) < 1.0001);
  }
  if (unit == 0) X.ms = INFINITY;
}

// firstOverSecond's size comparison (bvh_collision_traversal_node-inl.h:
// 77-89; OBBRSS::size = |OBB extents|^2, OBB-inl.h:206-209) from the FP32
// extents already loaded with the nodes.  Each FP32 sum of squares is
// within 5u (u = 2^-24) of the FP64 size, relative; outside a 50u band the
// FP32 order is the FP64 order, inside it (ties included) and for sizes
// near the FP32 underflow the FP64 sizes decide.  Saves the two scattered
// 8-B size loads of almost every descent.
__device__ __forceinline__ bool first_larger(const ObbNode32& n1, const ObbNode32& n2,
                                             const double* s1, const double* s2) {
  const float a = fmaf(n1.extent[2], n1.extent[2],
                       fmaf(n1.extent[1], n1.extent[1], n1.extent[0] * n1.extent[0]));
  const float b = fmaf(n2.extent[2], n2.extent[2],
                       fmaf(n2.extent[1], n2.extent[1], n2.extent[0] * n2.extent[0]));
  constexpr float kBand = 50.0f * 5.9604644775390625e-08f;
  if (a > 1e-30f && b > 1e-30f) {
    if (a > b * (1.0f + kBand)) return true;
    if (a < b * (1.0f - kBand)) return false;
  }
  return *s1 > *s2;
}

// A 64-B node record in four 16-B loads issued together (its child link
// with the rest, not in a later load once the cull has passed).
__device__ __forceinline__ ObbNode32 load_node32(const ObbNode32* p) {
  const uint4* w = reinterpret_cast<const uint4*>(p);
  const uint4 a = w[0], b = w[1], c = w[2], d = w[3];
  ObbNode32 n;
  uint4* o = reinterpret_cast<uint4*>(&n);
  o[0] = a;
  o[1] = b;
  o[2] = c;
  o[3] = d;
  return n;
}

// The query's 64-B FP32 transform record, likewise in four 16-B loads.
__device__ __forceinline__ QueryXf32 load_xf32(const QueryXf32* p) {
  static_assert(sizeof(QueryXf32) == 64, "four 16-B words");
  const uint4* w = reinterpret_cast<const uint4*>(p);
  const uint4 a = w[0], b = w[1], c = w[2], d = w[3];
  QueryXf32 x;
  uint4* o = reinterpret_cast<uint4*>(&x);
  o[0] = a;
  o[1] = b;
  o[2] = c;
  o[3] = d;
  return x;
}

}  // namespace fclx
