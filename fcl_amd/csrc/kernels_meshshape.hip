// Batched fcl::collide between a BVHModel<OBBRSS> and a primitive shape (Box,
// Sphere, Capsule, Cylinder, Convex) with FCL's GST_INDEP solver, in FP64:
//   orientedBVHShapeCollide (collision_func_matrix-inl.h:375-419, 500-521);
//   the shape's bounding box: computeBV<OBBRSS> by the generic fit over the
//   shape's bound vertices (geometry/shape/utility-inl.h:124-133, OBB fitn
//   bv/utility-inl.h:131-145), of which the BV test uses the OBB;
//   collisionRecurse (traversal_recurse-inl.h:82-129) over the mesh alone --
//   the shape is one leaf -- with BVTesting = OBB overlap of the shape's box
//   and the node's box posed by the mesh's transform
//   (mesh_shape_collision_traversal_node.h, OBBRSS node);
//   leaf test meshShapeCollisionOrientedNodeLeafTesting
//   (mesh_shape_collision_traversal_node-inl.h:205-283): sphereTriangleIntersect
//   (sphere_triangle-inl.h:138-230) for a sphere, GJK + EPA on the shape and
//   the posed TriangleP for the others (gjk_solver_indep-inl.h:448-505).
//
// One lane per query fits the shape's box (Jacobi eigenvectors of the bound
// vertices' covariance); then one wavefront per query descends the mesh in
// the reference's order (device/ordered.h) and stops at num_max_contacts.
// Without enable_contact a GJK "inside" is the answer (EPA's status is never
// Failed after it).  With it, GJK still decides the hit and the record's
// slot (count, cap and order are GJK's), and EPA only supplies the slot's
// contact: committed hits are queued and a second kernel runs GJK and EPA
// over the queue, each lane in a block of device memory of its own, taking
// the next queued pair when its own ends.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device/fit64.h"
#include "device/ordered.h"
#include "device/query32.h"
#include "device/shape64.h"
#include "kernels.h"

namespace fclx {

namespace {

constexpr int kBlk = 256;
constexpr int kMsListCap = 512;    // entries of a query's list in LDS
static_assert(kMsListDepth + 2 + 64 <= kMsListCap, "a tree path and a step");
// Lanes keep their pending right children in LDS up to this depth; in contexts
// with meshes deeper than MeshShapeLaunch::list_depth (up to kMsDeepMax levels) in device
// memory.
constexpr int kMsLaneStack = 64;
constexpr int kMsDeepMax = 4096;
constexpr int kMsDeepBlocksPerCu = 2;
constexpr int kEpaBlocksPerCu = 2;

// A hit whose contact EPA supplies: the query, the triangle and the record
// slot the contact goes to.
struct MsEpaSeed {
  int32_t q, prim;
  long long slot;
};

using shp::D3;
using shp::mk;


__device__ __forceinline__ double pick3(const double* a, int i) {
  return i == 0 ? a[0] : (i == 1 ? a[1] : a[2]);
}

// axisFromEigen (math/geometry-inl.h:561-598): columns = the eigenvectors of
// the largest and middle eigenvalues and their cross product.
__device__ void axis_from_eigen(const double E[9], const double s[3], double axis[9]) {
  int mn, mid, mx;
  if (s[0] > s[1]) {
    mx = 0;
    mn = 1;
  } else {
    mn = 0;
    mx = 1;
  }
  if (s[2] < pick3(s, mn)) {
    mid = mn;
    mn = 2;
  } else if (s[2] > pick3(s, mx)) {
    mid = mx;
    mx = 2;
  } else {
    mid = 2;
  }
  D3 c0, c1;
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    c0.v[r] = mx == 0 ? E[r] : (mx == 1 ? E[3 + r] : E[6 + r]);
    c1.v[r] = mid == 0 ? E[r] : (mid == 1 ? E[3 + r] : E[6 + r]);
  }
  const D3 c2 = shp::cross(c0, c1);
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    axis[3 * r + 0] = c0.v[r];
    axis[3 * r + 1] = c1.v[r];
    axis[3 * r + 2] = c2.v[r];
  }
}

// getBoundVertices in the shape's frame (box-inl.h:122-138,
// sphere-inl.h:96-120, capsule-inl.h:108-162, cylinder-inl.h:102-126); the
// same points in the same order.
__device__ int bound_points(const shp::Shape& s, D3* p) {
  switch (s.type) {
    case shp::kBox: {
      const double a = s.dims[0] / 2, b = s.dims[1] / 2, c = s.dims[2] / 2;
      int k = 0;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int l = 0; l < 2; ++l) p[k++] = mk(i ? -a : a, j ? -b : b, l ? -c : c);
      return 8;
    }
    case shp::kSphere: {
      const double m = (1 + sqrt(5.0)) / 2.0;
      const double e = s.dims[0] * 6 / (sqrt(27.0) + sqrt(15.0));
      const double a = e, b = m * e;
      p[0] = mk(0, a, b);
      p[1] = mk(0, -a, b);
      p[2] = mk(0, a, -b);
      p[3] = mk(0, -a, -b);
      p[4] = mk(a, b, 0);
      p[5] = mk(-a, b, 0);
      p[6] = mk(a, -b, 0);
      p[7] = mk(-a, -b, 0);
      p[8] = mk(b, 0, a);
      p[9] = mk(b, 0, -a);
      p[10] = mk(-b, 0, a);
      p[11] = mk(-b, 0, -a);
      return 12;
    }
    case shp::kCapsule: {
      const double r = s.dims[0], hl = s.dims[1] * 0.5;
      const double m = (1 + sqrt(5.0)) / 2.0;
      const double e = r * 6 / (sqrt(27.0) + sqrt(15.0));
      const double a = e, b = m * e, r2 = r * 2 / sqrt(3.0);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // b - hl written as b + (-hl): the same double
        const double z = h ? -hl : hl;
        D3* q = p + 12 * h;
        q[0] = mk(0, a, b + z);
        q[1] = mk(0, -a, b + z);
        q[2] = mk(0, a, -b + z);
        q[3] = mk(0, -a, -b + z);
        q[4] = mk(a, b, z);
        q[5] = mk(-a, b, z);
        q[6] = mk(a, -b, z);
        q[7] = mk(-a, -b, z);
        q[8] = mk(b, 0, a + z);
        q[9] = mk(b, 0, -a + z);
        q[10] = mk(-b, 0, a + z);
        q[11] = mk(-b, 0, -a + z);
      }
      const double c = 0.5 * r2, d = r;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double z = h ? -hl : hl;
        D3* q = p + 24 + 6 * h;
        q[0] = mk(r2, 0, z);
        q[1] = mk(c, d, z);
        q[2] = mk(-c, d, z);
        q[3] = mk(-r2, 0, z);
        q[4] = mk(-c, -d, z);
        q[5] = mk(c, -d, z);
      }
      return 36;
    }
    case shp::kCylinder: {
      const double r = s.dims[0], hl = s.dims[1] * 0.5;
      const double r2 = r * 2 / sqrt(3.0), a = 0.5 * r2, b = r;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double z = h ? hl : -hl;
        D3* q = p + 6 * h;
        q[0] = mk(r2, 0, z);
        q[1] = mk(a, b, z);
        q[2] = mk(-a, b, z);
        q[3] = mk(-r2, 0, z);
        q[4] = mk(-a, -b, z);
        q[5] = mk(a, -b, z);
      }
      return 12;
    }
  }
  return 0;
}

// The shape's box in the world frame: OBB fitn over the posed bound
// vertices (a convex's own vertices): point covariance
// (geometry-inl.h:1335-1421), eigen_old, axisFromEigen,
// getExtentAndCenter_pointcloud (geometry-inl.h:228-287).
__device__ void shape_obb(const shp::Shape& s, const shp::Xf& T, double axis[9], double to[3],
                          double extent[3]) {
  D3 local[36];
  const bool convex = s.type == shp::kConvex;
  const int n = convex ? s.nv : bound_points(s, local);
  double S1[3] = {0, 0, 0};
  double s00 = 0, s11 = 0, s22 = 0, s01 = 0, s02 = 0, s12 = 0;
  for (int i = 0; i < n; ++i) {
    const D3 q = convex ? mk(s.verts[3 * i], s.verts[3 * i + 1], s.verts[3 * i + 2]) : local[i];
    const D3 p = shp::apply(T, q);
#pragma unroll
    for (int k = 0; k < 3; ++k) S1[k] += p.v[k];
    s00 += p.v[0] * p.v[0];
    s11 += p.v[1] * p.v[1];
    s22 += p.v[2] * p.v[2];
    s01 += p.v[0] * p.v[1];
    s02 += p.v[0] * p.v[2];
    s12 += p.v[1] * p.v[2];
  }
  const double np = static_cast<double>(n);
  double M[9], E[9], ev[3];
  M[0] = s00 - S1[0] * S1[0] / np;
  M[4] = s11 - S1[1] * S1[1] / np;
  M[8] = s22 - S1[2] * S1[2] / np;
  M[1] = s01 - S1[0] * S1[1] / np;
  M[5] = s12 - S1[1] * S1[2] / np;
  M[2] = s02 - S1[0] * S1[2] / np;
  M[3] = M[1];
  M[6] = M[2];
  M[7] = M[5];
  eigen_old(M, ev, E);
  axis_from_eigen(E, ev, axis);
  double mn[3] = {1.7976931348623157e308, 1.7976931348623157e308, 1.7976931348623157e308};
  double mx[3] = {-1.7976931348623157e308, -1.7976931348623157e308, -1.7976931348623157e308};
  for (int i = 0; i < n; ++i) {
    const D3 q = convex ? mk(s.verts[3 * i], s.verts[3 * i + 1], s.verts[3 * i + 2]) : local[i];
    const D3 p = shp::apply(T, q);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double pr = shp::dot(shp::col(axis, k), p);
      if (pr > mx[k]) mx[k] = pr;
      if (pr < mn[k]) mn[k] = pr;
    }
  }
  const D3 o = mk((mx[0] + mn[0]) / 2, (mx[1] + mn[1]) / 2, (mx[2] + mn[2]) / 2);
  const D3 c = shp::rot(axis, o);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    to[k] = c.v[k];
    extent[k] = (mx[k] - mn[k]) * 0.5;
  }
}

// segmentSqrDistance (sphere_triangle-inl.h:84-108)
__device__ __forceinline__ double segment_sqr_distance(const D3& from, const D3& to, const D3& p,
                                                       D3& nearest) {
  D3 diff = shp::sub(p, from);
  const D3 v = shp::sub(to, from);
  double t = shp::dot(v, diff);
  if (t > 0) {
    const double dotVV = shp::dot(v, v);
    if (t < dotVV) {
      t /= dotVV;
      diff = shp::sub(diff, shp::mul(v, t));
    } else {
      t = 1;
      diff = shp::sub(diff, v);
    }
  } else {
    t = 0;
  }
  nearest = shp::add(from, shp::mul(v, t));
  return shp::dot(diff, diff);
}

// projectInTriangle (sphere_triangle-inl.h:112-135)
__device__ __forceinline__ bool project_in_triangle(const D3& p1, const D3& p2, const D3& p3,
                                                    const D3& n, const D3& p) {
  const double r1 = shp::dot(shp::cross(shp::sub(p2, p1), n), shp::sub(p, p1));
  const double r2 = shp::dot(shp::cross(shp::sub(p3, p2), n), shp::sub(p, p2));
  const double r3 = shp::dot(shp::cross(shp::sub(p1, p3), n), shp::sub(p, p3));
  return (r1 > 0 && r2 > 0 && r3 > 0) || (r1 <= 0 && r2 <= 0 && r3 <= 0);
}

// sphereTriangleIntersect (sphere_triangle-inl.h:138-230): the solver's
// outputs (normal from the centre towards the contact, depth <= 0).
__device__ bool sphere_triangle(double radius, const D3& center, const D3& P1, const D3& P2,
                                const D3& P3, D3& point, double& depth, D3& normal_out) {
  D3 normal = shp::normalized(shp::cross(shp::sub(P2, P1), shp::sub(P3, P1)));
  const double rt = radius + 2.220446049250313e-16;
  double dist = shp::dot(shp::sub(center, P1), normal);
  if (dist < 0) {
    dist *= -1;
    normal = shp::mul(normal, -1.0);
  }
  if (!(dist < rt)) return false;
  bool has = false;
  D3 cp = mk(0, 0, 0);
  if (project_in_triangle(P1, P2, P3, normal, center)) {
    has = true;
    cp = shp::sub(center, shp::mul(normal, dist));
  } else {
    const double r2 = rt * rt;
    D3 ne;
    if (segment_sqr_distance(P1, P2, center, ne) < r2) {
      has = true;
      cp = ne;
    }
    if (segment_sqr_distance(P2, P3, center, ne) < r2) {
      has = true;
      cp = ne;
    }
    if (segment_sqr_distance(P3, P1, center, ne) < r2) {
      has = true;
      cp = ne;
    }
  }
  if (!has) return false;
  const D3 cc = shp::sub(cp, center);
  const double dsq = shp::sqn(cc);
  if (!(dsq < rt * rt)) return false;
  if (dsq > 0) {
    normal_out = shp::normalized(cc);
    depth = -(radius - sqrt(dsq));
  } else {
    normal_out = shp::neg(normal);
    depth = -radius;
  }
  point = cp;
  return true;
}

// A usable query: a mesh of OBBRSS nodes no deeper than the stack (depth_max
// levels), and a shape of a known type (a convex with at least 4 vertices
// inside the pool).
__device__ __forceinline__ bool load_query(const MeshShapeLaunch& L, int q, shp::Shape& s,
                                           int depth_max) {
  const int mi = L.query_meshes[q], si = L.query_shapes[q];
  if (mi < 0 || mi >= L.num_meshes || si < 0 || si >= L.num_shapes) return false;
  const MeshDev& M = L.meshes[mi];
  if (M.num_bvs <= 0 || M.bv_type != 0 || M.depth > depth_max) return false;
  const fclx_shape& r = L.shapes[si];
  s.type = r.type;
  s.nv = r.num_vertices;
  s.dims[0] = r.dims[0];
  s.dims[1] = r.dims[1];
  s.dims[2] = r.dims[2];
  s.verts = nullptr;
  switch (r.type) {
    case shp::kBox:
    case shp::kSphere:
    case shp::kCapsule:
    case shp::kCylinder:
      return true;
    case shp::kConvex:
      if (r.num_vertices < 4 || r.vertex_offset < 0 ||
          r.vertex_offset + r.num_vertices > L.num_vertices || L.vertices == nullptr)
        return false;
      s.verts = L.vertices + 3 * r.vertex_offset;
      return true;
  }
  return false;
}

// For lanes: the queries grouped by shape kind, so that a wavefront's lanes run
// the same leaf test (their order does not change any query's answer).  Keys:
// the five kinds, 5 for a query whose mesh or shape id is out of range, and
// 6, last, for those of more than L.lanes_max nodes, which run on wavefronts.
// ctr[0..6]: counts, ctr[8..14]: placement cursors.
constexpr int kKinds = 7;

__device__ __forceinline__ int kind_of(const MeshShapeLaunch& L, int q) {
  const int mi = L.query_meshes[q], si = L.query_shapes[q];
  if (mi < 0 || mi >= L.num_meshes || si < 0 || si >= L.num_shapes) return 5;
  if (L.lanes_max != kAllLanes && L.meshes[mi].num_bvs > L.lanes_max) return 6;
  const int t = L.shapes[si].type;
  return t >= 0 && t < 5 ? t : 5;
}

__global__ void ms_zero(int32_t* ctr) {
  if (threadIdx.x < 16) ctr[threadIdx.x] = 0;
}

__global__ void __launch_bounds__(kBlk) ms_count(MeshShapeLaunch L, int32_t* ctr) {
  __shared__ int cnt[kKinds];
  if (threadIdx.x < kKinds) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int i = blockIdx.x * kBlk + threadIdx.x;
  if (i < L.num_queries) atomicAdd(&cnt[kind_of(L, i)], 1);
  __syncthreads();
  if (threadIdx.x < kKinds && cnt[threadIdx.x]) atomicAdd(&ctr[threadIdx.x], cnt[threadIdx.x]);
}

__global__ void __launch_bounds__(kBlk) ms_place(MeshShapeLaunch L, int32_t* ctr,
                                                 int32_t* order) {
  __shared__ int cnt[kKinds];
  __shared__ int base[kKinds];
  if (threadIdx.x < kKinds) cnt[threadIdx.x] = 0;
  __syncthreads();
  const int i = blockIdx.x * kBlk + threadIdx.x;
  int key = 0, off = 0;
  if (i < L.num_queries) {
    key = kind_of(L, i);
    off = atomicAdd(&cnt[key], 1);
  }
  __syncthreads();
  if (threadIdx.x < kKinds) {
    int start = 0;
    for (int k = 0; k < static_cast<int>(threadIdx.x); ++k) start += ctr[k];
    base[threadIdx.x] =
        start + (cnt[threadIdx.x] ? atomicAdd(&ctr[8 + threadIdx.x], cnt[threadIdx.x]) : 0);
  }
  __syncthreads();
  if (i < L.num_queries) order[base[key] + off] = i;
}

// The leaf test of one (shape, triangle) pair, kept out of line so that the
// descent loop's registers are not sized for GJK and EPA.
template <bool kContact>
__device__ __noinline__ bool leaf_test(const shp::Shape& s, const shp::Xf& T1, const shp::Xf& T2,
                                       const double* tv, double tol, shp::Epa& E,
                                       shp::Contact& c) {
  bool hit;
  if (s.type == shp::kSphere) {
    // gjk_solver_indep-inl.h:527-545: the triangle posed by the mesh's tf
    D3 P[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) P[k] = shp::apply(T1, mk(tv[3 * k], tv[3 * k + 1], tv[3 * k + 2]));
    D3 p, n;
    double d;
    hit = sphere_triangle(s.dims[0], T2.t, P[0], P[1], P[2], p, d, n);
    if (hit) {
      c.pos = p;
      c.normal = shp::neg(n);  // the leaf stores minus the solver's normal
      c.depth = d;
    }
  } else {
    shp::Shape tri;
    tri.type = shp::kTriangle;
    tri.nv = 3;
    tri.dims[0] = tri.dims[1] = tri.dims[2] = 0;
    tri.verts = tv;
    shp::MDiff m;
    shp::make_mdiff(s, T2, tri, T1, m);
    shp::Gjk g;
    hit = shp::gjk_evaluate(g, m, tol) == shp::kGjkInside;
    if constexpr (kContact) {
      if (hit) {
        // the leaf's -normal undoes the solver's: EPA's normal stays
        bool more = shp::epa_start(E, g, m, tol);
        while (more) more = shp::epa_step(E, m, tol);
        c = shp::epa_finish(E, m, T2);
      }
    }
  }
  return hit;
}

// One query of the group traversal, prepared by one lane.
struct alignas(128) MsQuery {
  double axis[9], to[3], ext[3];  // the shape's box in the world frame
  int32_t valid;
  int32_t unit;                   // the mesh's rotation and the box axes are unit vectors:
                                  // the FP32 cull's margin holds
};
static_assert(sizeof(MsQuery) == 128, "one line per query");

__global__ void __launch_bounds__(kBlk) meshshape_setup(MeshShapeLaunch L, MsQuery* out) {
  const int q = blockIdx.x * kBlk + threadIdx.x;
  if (q >= L.num_queries) return;
  if (L.lanes_max > 0 && kind_of(L, q) != 6) return;  // a lane's
  MsQuery r;
  shp::Shape s;
  r.valid = load_query(L, q, s, L.max_depth) ? 1 : 0;
  r.unit = 0;
  if (r.valid) {
    shape_obb(s, shp::xf_load(L.tf2 + 12 * static_cast<size_t>(q)), r.axis, r.to, r.ext);
    const double* R = L.tf1 + 12 * static_cast<size_t>(q);
    bool unit = true;
#pragma unroll
    for (int k = 0; k < 3; ++k)
      unit = unit && sq(col(R, k)) < 1.0001 && sq(v3(R[3 * k], R[3 * k + 1], R[3 * k + 2])) < 1.0001 &&
             sq(col(r.axis, k)) < 1.0001;
    r.unit = unit ? 1 : 0;
  } else {
    L.counts[q] = 0;
    if (L.stats) {
      L.stats[2 * q] = 0;
      L.stats[2 * q + 1] = 0;
    }
    atomicOr(L.status, kStatusBadQuery);
  }
  out[q] = r;
}

// A group's query in LDS.
struct MsWave {
  shp::Shape s;
  shp::Xf T1, T2;
  MsQuery m;
  QueryXf32 x32;   // the mesh's pose, with the cull's margin
  ObbNode32 box32; // the shape's box
  const ObbNode32* n32;
  const ObbNode64* n64;
  const double* tris;
};

// The leaf test's answer alone: a sphere by the closed form, the other
// shapes by GJK.
__device__ __forceinline__ bool leaf_inside(const MsWave& w, const double* tv, double tol) {
  if (w.s.type == shp::kSphere) {
    D3 P[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      P[k] = shp::apply(w.T1, mk(tv[3 * k], tv[3 * k + 1], tv[3 * k + 2]));
    D3 p, n;
    double d;
    return sphere_triangle(w.s.dims[0], w.T2.t, P[0], P[1], P[2], p, d, n);
  }
  shp::Shape tri;
  tri.type = shp::kTriangle;
  tri.nv = 3;
  tri.dims[0] = tri.dims[1] = tri.dims[2] = 0;
  tri.verts = tv;
  shp::MDiff m;
  shp::make_mdiff(w.s, w.T2, tri, w.T1, m);
  shp::Gjk g;
  return shp::gjk_evaluate(g, m, tol) == shp::kGjkInside;
}

// collide(mesh, shape) in the reference's order (device/ordered.h), one
// wavefront per query: FP32 certified culls of the mesh's nodes against the
// shape's box (FP64 where unsure), leaf tests once leaf_min leaf entries
// have gathered or nothing else is left to test.  With contacts, a committed
// hit takes its record slot; spheres write their contact at once, the others
// are queued for EPA.
//
// Bound: GJK, about 75 us for a round of up to 64 at two wavefronts per SIMD
// (two thirds of the kernel), whatever the number of lanes in it; so a
// round waits for a full wavefront of leaves (leaf_min 64; 100,000 links
// around 20,480 triangles, 258 nodes and 79 leaves on average and up to
// 20,713 and 9,888: 11.1 ms, at 32 14.1 ms, at 16 19.4 ms).  One lane per
// query, as before, took 330-460 ms for this batch, the time of its longest
// query; 200,000 links that nearly all collide at once 8.3 ms, now 7.3.
// Quarter wavefronts are faster for the latter (4.2 ms) and slower for the
// former (28 ms).  Large batches on small meshes run on lanes (below).
template <bool kStats, bool kContact>
__device__ __forceinline__ void descend(const MeshShapeLaunch& L, const MsQuery* queries, size_t q,
                                        int margin, int leaf_min, MsEpaSeed* seeds,
                                        unsigned long long* nseed,
                                        OrderedList<kMsListCap, kStats>& S, MsWave& w) {
  constexpr int G = 64, kCap = kMsListCap;
  const LaneGroup<G> g;
  if (queries[q].valid == 0) return;
  OrdTotals T = ord_begin(g, S, 0u);
  if (g.lane == 0) {
    const MeshDev& M = L.meshes[L.query_meshes[q]];
    (void)load_query(L, static_cast<int>(q), w.s, L.max_depth);
    w.T1 = shp::xf_load(L.tf1 + 12 * q);
    w.T2 = shp::xf_load(L.tf2 + 12 * q);
    const MsQuery m = queries[q];
    w.m = m;
    QueryXf32 X;
    make_xf32(w.T1.R, w.T1.t.v, (fabs(m.to[0]) + fabs(m.to[1])) + fabs(m.to[2]), M.cmax, X);
    if (!m.unit) X.ms = INFINITY;  // every test is left to FP64
    X.m1 = X.m2 = 0;
    X.valid = 1;
    w.x32 = X;
    ObbNode32 b;
#pragma unroll
    for (int k = 0; k < 9; ++k) b.axis[k] = static_cast<float>(m.axis[k]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      b.to[k] = static_cast<float>(m.to[k]);
      b.extent[k] = static_cast<float>(m.ext[k]);
    }
    b.first_child = 0;
    w.box32 = b;
    w.n32 = M.obb32;
    w.n64 = M.obb64;
    w.tris = M.tri_verts;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  while (T.sp > 0) {
    // (a query tests no node twice: its counts fit the list's 32 bits)
    const int n = ord_window<G, kCap>(T.sp, margin);
    const bool on = g.lane < n;
    unsigned long long e = 0;
    uint2 acc = make_uint2(0u, 0u);
    if (on) {
      e = S.e[T.sp - 1 - g.lane];
      if constexpr (kStats) acc = S.acc[T.sp - 1 - g.lane];
    }
    const int kind = ord_kind(e), id = ord_a(e);
    const bool node = on && kind == kOrdNode, leaf = on && kind == kOrdLeaf;
    OrdOutcome r;
    if (on && kind >= kOrdHit) {
      r.nout = 1;
      r.o0 = e;
      r.hit = true;
      r.n = 1;
    }
    const unsigned long long lm = __ballot(leaf);
    const bool test_leaves = lm != 0 && (__popcll(lm) >= leaf_min || __ballot(node) == 0);
    if (node) {
      const ObbNode32 nd = load_node32(w.n32 + id);
      r.bv = 1;
      int c = obb_cull32(w.x32, w.box32, nd);
      if (c == kCullUnsure) {
        const ObbNode64& n64 = w.n64[id];
        M3 R0;
#pragma unroll
        for (int i = 0; i < 9; ++i) R0.m[i] = w.T1.R[i];
        double B[9], Tr[3];
        box_relative(R0, v3(w.T1.t.v[0], w.T1.t.v[1], w.T1.t.v[2]), w.m.axis, w.m.to, n64.axis,
                     n64.to, B, Tr);
        c = obb_disjoint64(B, Tr, w.m.ext, n64.extent) ? kCullDisjoint : kCullOverlap;
      }
      if (c == kCullOverlap) {
        const int fc = nd.first_child;
        if (fc >= 0) {
          r.nout = 2;
          r.o0 = ord_pack(kOrdNode, fc, 0);
          r.o1 = ord_pack(kOrdNode, fc + 1, 0);
        } else {
          r.nout = 1;
          r.o0 = ord_pack(kOrdLeaf, -(fc + 1), 0);
        }
      }
    } else if (leaf) {
      if (test_leaves) {
        r.leaf = 1;
        if (leaf_inside(w, w.tris + static_cast<size_t>(id) * kTriVertsStride, L.tol)) {
          r.nout = 1;
          r.hit = true;
          r.n = 1;
          r.o0 = ord_pack(kOrdHit + 1, id, 0);
        }
      } else {
        r.nout = 1;
        r.o0 = e;
      }
    }
    ord_settle<G, kCap, kStats>(g, S, T, r, acc, n, L.cap, [&](bool mine, int take, int before,
                                                               int total) {
      (void)total;
      const bool store = mine && take > 0;
      const size_t slot = q * L.cap + T.count + before;
      const int prim = ord_a(r.o0);
      if (store && L.prims) L.prims[slot] = prim;
      if constexpr (kContact) {
        const bool sphere = w.s.type == shp::kSphere;
        const unsigned long long em = __ballot(store && !sphere);
        if (em != 0) {  // one reservation for the wavefront
          const int leader = __ffsll(static_cast<long long>(em)) - 1;
          unsigned long long b = 0;
          if (static_cast<int>(__lane_id()) == leader)
            b = atomicAdd(nseed, static_cast<unsigned long long>(__popcll(em)));
          b = __shfl(b, leader);
          if (store && !sphere)
            seeds[b + __popcll(em & ((1ULL << __lane_id()) - 1ULL))] =
                MsEpaSeed{static_cast<int32_t>(q), prim, static_cast<long long>(slot)};
        }
        if (store && sphere) {
          const double* tv = w.tris + static_cast<size_t>(prim) * kTriVertsStride;
          D3 P[3];
#pragma unroll
          for (int k = 0; k < 3; ++k)
            P[k] = shp::apply(w.T1, mk(tv[3 * k], tv[3 * k + 1], tv[3 * k + 2]));
          D3 p, nn;
          double d;
          (void)sphere_triangle(w.s.dims[0], w.T2.t, P[0], P[1], P[2], p, d, nn);
          nn = shp::neg(nn);  // the leaf stores minus the solver's normal
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            L.contact_pos[3 * slot + j] = p.v[j];
            L.contact_normal[3 * slot + j] = nn.v[j];
          }
          L.contact_depth[slot] = d;
        }
      }
    });
  }
  if (g.lane == 0) {
    L.counts[q] = T.count;
    if constexpr (kStats) {
      L.stats[2 * q] = S.total.x;
      L.stats[2 * q + 1] = S.total.y;
    }
  }
}

// A block per query from `first` on (a loop over queries took 1 % of a batch);
// kSome: the last part of an order, whose other queries are the lanes'.
template <bool kStats, bool kContact, int kWaves, bool kSome>
__global__ void __launch_bounds__(64, kWaves) meshshape_ordered(MeshShapeLaunch L,
                                                                const MsQuery* queries, int margin,
                                                                int leaf_min, MsEpaSeed* seeds,
                                                                unsigned long long* nseed,
                                                                int first, const int32_t* order,
                                                                const int32_t* ctr) {
  __shared__ OrderedList<kMsListCap, kStats> S;
  __shared__ MsWave w;
  if constexpr (kSome) {
    const size_t end = L.num_queries;
    for (size_t k = end - static_cast<size_t>(ctr[6]) + blockIdx.x; k < end; k += gridDim.x)
      descend<kStats, kContact>(L, queries, static_cast<size_t>(order[k]), margin, leaf_min, seeds,
                                nseed, S, w);
  } else {
    descend<kStats, kContact>(L, queries, static_cast<size_t>(first) + blockIdx.x, margin, leaf_min,
                              seeds, nseed, S, w);
  }
}

// A query per lane.  Lanes of a wavefront step together: a lane whose descent
// reached a leaf that passed its BV test waits there, the others keep
// descending, and the waiting lanes test their leaves together once they are a
// set share of the live lanes (or nobody can descend).  The costly leaf test
// (GJK) then runs once for many lanes instead of once per descent step.  Each
// lane's own order of tests is the reference's, so counts, triangles and test
// statistics are unchanged.
//
// For the light queries of large batches (order: those grouped by kind, ctr:
// the groups' counts; the rule is at mesh_shape_lanes_max), whose hits are queued
// for EPA; and for what the lists in LDS do not hold: contexts with a mesh
// deeper than L.list_depth, and contact batches whose EPA queue would exceed
// its budget (EPA then runs in the descending lane).
//
// kDeep: the pending right children live in device memory (deep_stack, one
// column of L.max_depth entries per lane, lane-interleaved) instead of LDS.
template <bool kContact, bool kDeep, bool kQueue>
__global__ void __launch_bounds__(kBlk, kDeep ? 1 : 2) meshshape_lanes(
    MeshShapeLaunch L, const int32_t* order, const int32_t* ctr, shp::EpaLane* lanes,
    shp::EpaWave* waves, int* deep_stack, MsEpaSeed* seeds, unsigned long long* nseed) {
  constexpr bool kEpaHere = kContact && !kQueue;
  const size_t gid = static_cast<size_t>(blockIdx.x) * kBlk + threadIdx.x;
  const size_t stride = static_cast<size_t>(gridDim.x) * kBlk;
  const size_t end = static_cast<size_t>(L.num_queries) - (order ? static_cast<size_t>(ctr[6]) : 0);
  // the horizon walk's stack in LDS, one column per thread
  __shared__ int16_t xs_lds[kEpaHere ? shp::kNfEpa : 1][kBlk];
  shp::Epa E;
  if constexpr (kEpaHere) {
    E.M = lanes + gid;
    E.S = waves + gid / 64;
    E.lane = threadIdx.x & 63;
    E.xs = &xs_lds[0][threadIdx.x];
    E.xs_stride = kBlk;
  }
  size_t qq = gid;  // position in the order
  size_t q = 0;     // the query at that position
  shp::Shape s;
  shp::Xf T1, T2;
  double sa[9], sto[3], sext[3];
  const ObbNode64* nodes = nullptr;
  const double* tris = nullptr;
  // pending right children in LDS, one column per lane (lane-interleaved:
  // conflict-free whatever depth each lane is at)
  __shared__ int stk[kDeep ? 1 : kMsLaneStack][kBlk];
  const int column = threadIdx.x;
  int sp = 0, b = 0, count = 0, pend = -1;
  long long nbv = 0, nleaf = 0;
  bool live = false;  // a query in progress
  auto push = [&](int v) {
    if constexpr (kDeep)
      deep_stack[static_cast<size_t>(sp) * stride + gid] = v;
    else
      stk[sp][column] = v;
    ++sp;
  };
  auto pop = [&]() -> int {
    --sp;
    if constexpr (kDeep)
      return deep_stack[static_cast<size_t>(sp) * stride + gid];
    else
      return stk[sp][column];
  };
  // take queries until one is usable (the others are answered at once)
  auto start = [&]() {
    while (qq < end) {
      q = order ? static_cast<size_t>(order[qq]) : qq;
      if (load_query(L, static_cast<int>(q), s, L.max_depth)) {
        const MeshDev& M = L.meshes[L.query_meshes[q]];
        nodes = M.obb64;
        tris = M.tri_verts;
        T1 = shp::xf_load(L.tf1 + 12 * q);
        T2 = shp::xf_load(L.tf2 + 12 * q);
        shape_obb(s, T2, sa, sto, sext);
        sp = 0;
        b = 0;
        count = 0;
        pend = -1;
        nbv = 0;
        nleaf = 0;
        live = true;
        return;
      }
      L.counts[q] = 0;
      if (L.stats) {
        L.stats[2 * q] = 0;
        L.stats[2 * q + 1] = 0;
      }
      atomicOr(L.status, kStatusBadQuery);
      qq += stride;
    }
    live = false;
  };
  auto finish = [&]() {
    L.counts[q] = count;
    if (L.stats) {
      L.stats[2 * q] = nbv;
      L.stats[2 * q + 1] = nleaf;
    }
    qq += stride;
    start();
  };
  auto next = [&]() {  // the next node of the descent, or the query's end
    if (sp == 0)
      finish();
    else
      b = pop();
  };
  start();
  while (true) {
    const bool walk = live && pend < 0;
    const unsigned long long mw = __ballot(walk);
    const unsigned long long ml = __ballot(live && pend >= 0);
    if (!mw && !ml) break;
    if (ml && (!mw || 100 * __popcll(ml) >= L.leaf_share * __popcll(mw | ml))) {
      if (pend < 0) continue;
      const int prim = pend;
      pend = -1;
      ++nleaf;
      shp::Contact c;
      const bool hit =
          leaf_test<kEpaHere>(s, T1, T2, tris + static_cast<size_t>(prim) * kTriVertsStride, L.tol,
                              E, c);
      const bool queued = kQueue && s.type != shp::kSphere;
      if constexpr (kQueue) {
        // the hits of this leaf round for EPA: one reservation for the wavefront
        const unsigned long long em = __ballot(hit && queued);
        if (em != 0) {
          const int leader = __ffsll(static_cast<long long>(em)) - 1;
          unsigned long long at = 0;
          if (static_cast<int>(threadIdx.x & 63) == leader)
            at = atomicAdd(nseed, static_cast<unsigned long long>(__popcll(em)));
          at = __shfl(at, leader);
          if (hit && queued)
            seeds[at + __popcll(em & ((1ULL << (threadIdx.x & 63)) - 1ULL))] = MsEpaSeed{
                static_cast<int32_t>(q), prim, static_cast<long long>(q * L.cap + count)};
        }
      }
      if (hit) {
        const size_t k = q * L.cap + count;
        if (L.prims) L.prims[k] = prim;
        if constexpr (kContact) {
          if (!queued) {
#pragma unroll
            for (int j = 0; j < 3; ++j) {
              L.contact_pos[3 * k + j] = c.pos.v[j];
              L.contact_normal[3 * k + j] = c.normal.v[j];
            }
            L.contact_depth[k] = c.depth;
          }
        }
        if (++count >= L.cap) {
          finish();
          continue;
        }
      }
      next();
    } else if (walk) {
      const ObbNode64& nd = nodes[b];
      ++nbv;
      M3 R0;
#pragma unroll
      for (int i = 0; i < 9; ++i) R0.m[i] = T1.R[i];
      double B[9], Tr[3];
      box_relative(R0, v3(T1.t.v[0], T1.t.v[1], T1.t.v[2]), sa, sto, nd.axis, nd.to, B, Tr);
      if (obb_disjoint64(B, Tr, sext, nd.extent)) {
        next();
      } else if (nd.first_child >= 0) {
        push(nd.first_child + 1);
        b = nd.first_child;
      } else {
        pend = -(nd.first_child + 1);  // tested in the next leaf round
      }
    }
  }
}

// EPA over the queued hits, each lane on its own pair one EPA loop pass per
// trip, taking the wavefront's next entry when its own ends (the entries
// come 64 at a time per wavefront from one counter), so that lanes do not
// wait for the slowest pair of their wavefront.  The contact goes to the
// slot the descent reserved, as leaf_test<true> writes it.
template <int kWaves>
__global__ void __launch_bounds__(kBlk, kWaves) meshshape_epa(MeshShapeLaunch L,
                                                              const MsEpaSeed* seeds,
                                                              const unsigned long long* nseed,
                                                              unsigned long long* grab,
                                                              shp::EpaLane* lanes,
                                                              shp::EpaWave* waves) {
  constexpr int kRefillAt = 16;
  const int lane = threadIdx.x & 63;
  const size_t gid = static_cast<size_t>(blockIdx.x) * kBlk + threadIdx.x;
  const long long total = static_cast<long long>(*nseed);
  long long cursor = 0, stop = 0;  // the wavefront's entries not yet started
  bool exhausted = total == 0;
  __shared__ int16_t xs_lds[shp::kNfEpa][kBlk];  // the horizon walk's stack
  shp::Epa E;
  E.M = lanes + gid;
  E.S = waves + gid / 64;
  E.lane = lane;
  E.xs = &xs_lds[0][threadIdx.x];
  E.xs_stride = kBlk;
  shp::MDiff m;
  shp::Xf T2;
  long long slot = 0;
  bool active = false;
  while (true) {
    bool finish = false, started = false;
    const unsigned long long idle = __ballot(!active);
    const int nidle = __popcll(idle);
    if (cursor >= stop && !exhausted && (nidle == 64 || nidle >= kRefillAt)) {
      unsigned long long base = 0;
      if (lane == 0) base = atomicAdd(grab, 64ULL);
      base = __shfl(base, 0);
      const long long b = static_cast<long long>(base);
      cursor = b < total ? b : total;
      stop = b + 64 < total ? b + 64 : total;
      exhausted = b + 64 >= total;
    }
    if (cursor < stop && (nidle == 64 || nidle >= kRefillAt)) {
      const long long v = cursor + __popcll(idle & ((1ULL << lane) - 1ULL));
      cursor = cursor + nidle < stop ? cursor + nidle : stop;
      if (!active && v < stop) {
        const MsEpaSeed& sd = seeds[v];
        const int q = sd.q;
        shp::Shape s;
        (void)load_query(L, q, s, kMsDeepMax);  // checked by the descent
        const MeshDev& M = L.meshes[L.query_meshes[q]];
        shp::Shape tri;
        tri.type = shp::kTriangle;
        tri.nv = 3;
        tri.dims[0] = tri.dims[1] = tri.dims[2] = 0;
        tri.verts = M.tri_verts + static_cast<size_t>(sd.prim) * kTriVertsStride;
        const shp::Xf T1 = shp::xf_load(L.tf1 + 12 * static_cast<size_t>(q));
        T2 = shp::xf_load(L.tf2 + 12 * static_cast<size_t>(q));
        shp::make_mdiff(s, T2, tri, T1, m);
        // GJK once more, for its final simplex ("inside", as the descent found)
        shp::Gjk g;
        (void)shp::gjk_evaluate(g, m, L.tol);
        slot = sd.slot;
        active = shp::epa_start(E, g, m, L.tol);
        finish = !active;
        started = true;
      }
    }
    if (active && !started) {
      active = shp::epa_step(E, m, L.tol);
      finish = !active;
    }
    if (finish) {
      // the leaf's -normal undoes the solver's: EPA's normal stays
      const shp::Contact c = shp::epa_finish(E, m, T2);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        L.contact_pos[3 * slot + j] = c.pos.v[j];
        L.contact_normal[3 * slot + j] = c.normal.v[j];
      }
      L.contact_depth[slot] = c.depth;
    }
    if (exhausted && cursor >= stop && !__ballot(active)) break;
  }
}

}  // namespace

size_t mesh_shape_epa_lane_bytes() { return sizeof(shp::EpaLane) + sizeof(shp::EpaWave) / 64; }

__global__ void ms_zero_u64(unsigned long long* p) {
  if (threadIdx.x < 2) p[threadIdx.x] = 0;
}

namespace {

template <int kWaves, bool kSome>
void launch_descent(const MeshShapeLaunch& L, const MsQuery* queries, MsEpaSeed* seeds,
                    unsigned long long* nseed, const int32_t* order, const int32_t* ctr,
                    hipStream_t s) {
  auto kernel = L.contact ? (L.stats ? meshshape_ordered<true, true, kWaves, kSome>
                                     : meshshape_ordered<false, true, kWaves, kSome>)
                          : (L.stats ? meshshape_ordered<true, false, kWaves, kSome>
                                     : meshshape_ordered<false, false, kWaves, kSome>);
  const int leaf_min = L.leaf_share > 0 ? std::max(1, 64 * L.leaf_share / 100) : 64;
  // HIP refuses a launch of 2^32 threads
  constexpr int kPart = 1 << 25;
  for (long long first = 0; first < L.num_queries; first += kPart) {
    const long long left = L.num_queries - first;
    const unsigned blocks =
        kSome ? group_blocks(left) : static_cast<unsigned>(std::min<long long>(left, kPart));
    kernel<<<blocks, 64, 0, s>>>(L, queries, L.max_depth + 2, leaf_min, seeds, nseed,
                                 static_cast<int>(first), order, ctr);
    if (kSome) return;
  }
}

// Leaf rounds of the lanes, measured: at half the live lanes for booleans, three
// quarters with contact geometry.
int lane_leaf_share(const MeshShapeLaunch& L) {
  return L.leaf_share > 0 ? L.leaf_share : (L.contact ? 75 : 50);
}

// Stream-ordered scratch of one batch, freed (in stream order) at its end.
struct StreamScratch {
  hipStream_t s;
  void* held[8] = {};
  int n = 0;
  explicit StreamScratch(hipStream_t stream) : s(stream) {}
  ~StreamScratch() {
    for (int i = 0; i < n; ++i) (void)hipFreeAsync(held[i], s);
  }
  template <typename T>
  hipError_t get(T** p, size_t count) {
    void* v = nullptr;
    const hipError_t e = hipMallocAsync(&v, std::max<size_t>(count * sizeof(T), 16), s);
    if (e == hipSuccess) {
      held[n++] = v;
      *p = static_cast<T*>(v);
    }
    return e;
  }
};

#define MS_TRY(expr)                     \
  do {                                   \
    const hipError_t e_ = (expr);        \
    if (e_ != hipSuccess) return e_;     \
  } while (0)

hipError_t launch_deep(MeshShapeLaunch L, int cus, hipStream_t s) {
  L.leaf_share = lane_leaf_share(L);
  long long grid = (static_cast<long long>(L.num_queries) + kBlk - 1) / kBlk;
  grid = std::min<long long>(grid, static_cast<long long>(cus) * kMsDeepBlocksPerCu);
  const size_t lanes = static_cast<size_t>(grid) * kBlk;
  StreamScratch mem(s);
  int* stack = nullptr;
  MS_TRY(mem.get(&stack, lanes * L.max_depth));
  shp::EpaLane* el = nullptr;
  shp::EpaWave* ew = nullptr;
  if (L.contact) {
    MS_TRY(mem.get(&el, lanes));
    MS_TRY(mem.get(&ew, lanes / 64));
  }
  auto kernel = L.contact ? meshshape_lanes<true, true, false> : meshshape_lanes<false, true, false>;
  kernel<<<static_cast<unsigned>(grid), kBlk, 0, s>>>(L, nullptr, nullptr, el, ew, stack, nullptr,
                                                      nullptr);
  return hipGetLastError();
}

// The queries of L.lanes_max nodes at most (all with kAllLanes) on a lane each.
// order, ctr: filled for launch_descent to take the others from.
hipError_t launch_lanes(MeshShapeLaunch L, MsEpaSeed* seeds, unsigned long long* nseed,
                        int32_t* order, int32_t* ctr, hipStream_t s) {
  L.leaf_share = lane_leaf_share(L);
  const unsigned grid = static_cast<unsigned>((L.num_queries + kBlk - 1) / kBlk);
  ms_zero<<<1, 64, 0, s>>>(ctr);
  ms_count<<<grid, kBlk, 0, s>>>(L, ctr);
  ms_place<<<grid, kBlk, 0, s>>>(L, ctr, order);
  auto kernel = L.contact ? meshshape_lanes<true, false, true> : meshshape_lanes<false, false, false>;
  kernel<<<grid, kBlk, 0, s>>>(L, order, ctr, nullptr, nullptr, nullptr, seeds, nseed);
  return hipGetLastError();
}

}  // namespace

// Where a lane per query is the faster form: on small meshes, in batches large
// enough to hide the lanes' waiting for each other's leaf rounds, which grows
// with the mesh (and with the contacts asked for).  Lanes / wavefronts, to the
// first hit: a triangle, 32,768 queries 249 / 314 us and 1,000,000 1.0 / 5.8 ms;
// 12 triangles 100,000 1.4 / 1.2, 131,072 1.4 / 1.4 and 1,000,000 4.6 / 10.3; 80
// triangles 131,072 2.74 / 2.68 and 250,000 3.6 / 5.0; 180 triangles 250,000 5.9 /
// 5.8; 320 triangles 500,000 12.2 / 12.4 and 1,000,000 20 / 25; 800 triangles
// 3,000,000 87 / 79.  To 4 hits: 80 triangles 131,072 3.7 / 2.7 and 250,000 4.8 /
// 5.0; 180 triangles 500,000 10.4 / 11.4; 320 triangles 1,000,000 26 / 25 and
// 3,000,000 67 / 71.
long long mesh_shape_lanes_max(int num_queries, int cap, size_t nodes_min, size_t nodes_max) {
  long long limit = num_queries >= 24576 ? 1 : 0;
  const long long over = num_queries >= 122880 ? (num_queries - 90112LL) / (cap > 1 ? 3 : 1) : 0;
  while (limit < 1023 && (limit + 1) * (limit + 1) <= over) ++limit;
  if (static_cast<long long>(nodes_min) > limit) return 0;
  return static_cast<long long>(nodes_max) <= limit ? kAllLanes : limit;
}

hipError_t launch_mesh_shape_collide(const MeshShapeLaunch& in, int waves, hipStream_t s) {
  if (in.num_queries <= 0) return hipSuccess;
  MeshShapeLaunch L = in;
  L.max_depth = std::min(L.max_depth, kMsDeepMax);  // deeper meshes are refused by load_query
  int dev = 0, cus = 0;
  MS_TRY(hipGetDevice(&dev));
  MS_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const size_t nslots = static_cast<size_t>(L.num_queries) * static_cast<size_t>(L.cap);
  if (L.max_depth > L.list_depth || (L.contact && nslots > L.epa_queue / sizeof(MsEpaSeed)))
    return launch_deep(L, cus, s);
  if (L.max_depth > kMsLaneStack) L.lanes_max = 0;
  StreamScratch mem(s);
  MsQuery* queries = nullptr;
  MsEpaSeed* seeds = nullptr;
  unsigned long long* ctr = nullptr;  // [0] seeds queued, [1] seeds handed out
  int32_t* order = nullptr;
  int32_t* kinds = nullptr;
  if (L.contact) {
    MS_TRY(mem.get(&seeds, nslots));
    MS_TRY(mem.get(&ctr, 2));
    ms_zero_u64<<<1, 64, 0, s>>>(ctr);
  }
  if (L.lanes_max > 0) {
    MS_TRY(mem.get(&order, static_cast<size_t>(L.num_queries)));
    MS_TRY(mem.get(&kinds, 16));
    MS_TRY(launch_lanes(L, seeds, ctr, order, kinds, s));
  }
  if (L.lanes_max != kAllLanes) {
    MS_TRY(mem.get(&queries, static_cast<size_t>(L.num_queries)));
    meshshape_setup<<<static_cast<unsigned>((L.num_queries + kBlk - 1) / kBlk), kBlk, 0, s>>>(
        L, queries);
    auto descent = order ? launch_descent<2, true>
                         : (waves == 1 ? launch_descent<1, false>
                                       : (waves == 3 ? launch_descent<3, false>
                                                     : launch_descent<2, false>));
    descent(L, queries, seeds, ctr, order, kinds, s);
  }
  MS_TRY(hipGetLastError());
  if (!L.contact) return hipSuccess;
  const long long egrid = static_cast<long long>(cus) * kEpaBlocksPerCu;
  const size_t lanes = static_cast<size_t>(egrid) * kBlk;
  StreamScratch emem(s);
  shp::EpaLane* el = nullptr;
  shp::EpaWave* ew = nullptr;
  MS_TRY(emem.get(&el, lanes));
  MS_TRY(emem.get(&ew, lanes / 64));
  meshshape_epa<2><<<static_cast<unsigned>(egrid), kBlk, 0, s>>>(L, seeds, ctr, ctr + 1, el, ew);
  return hipGetLastError();
}

}  // namespace fclx
