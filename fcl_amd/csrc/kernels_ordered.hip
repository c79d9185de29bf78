// collide() in the reference's order by lane groups (device/ordered.h): the
// single-query calls, contact geometry, small num_max_contacts and the
// re-run of queries that reached their cap.
//
// Each wavefront step loads the two 64-B FP32 nodes of up to 64 BVTT nodes,
// runs the certified FP32 cull (FP64 where it is unsure) and, once enough
// overlapping leaf pairs have gathered, the FP64 triangle tests.  Answers,
// their order and the test counts are those of collisionRecurse
// (traversal_recurse-inl.h:82-129), whatever was tested ahead.
//
// Bound: the latency of the step (pop from LDS, two node loads, the cull)
// times a query's longest chain of steps; a batch of lanes that each walk a
// whole query (one lane per query, the form before) waits for its longest
// query, up to 2,353 dependent visits where the mean is 287.  Measured,
// 2 x 2,420 triangles: 10,000 queries to their first contact 3.5 ms with a
// lane per query, 0.21 ms with a wavefront; 4,096 queries to 8 contacts with
// geometry 9.4 -> 0.26 ms; one collide() call 440 -> 72 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "device/ordered.h"
#include "device/query32.h"
#include "kernels.h"

namespace fclx {

namespace {

constexpr int kWave = 64;

// List entries per group.  A group of 64 serves every hierarchy the
// traversals take (summed depth <= kMaxStack) with room for full steps.
template <int G>
constexpr int list_cap() {
  return G == 64 ? 512 : 192;
}

// Batches to the first contact from this size on run four queries per
// wavefront: the chip is full either way, and a group of 16 tests less ahead
// of a query's answer.  1,000,000 queries of 2 x 2,420 triangles 15.5 ms by
// whole wavefronts, 8.7 ms by quarters; 10,000 queries 0.23 against 0.37 ms.
// With statistics 65,536 queries 1.31 against 1.17 and 1,000,000 18.4 against
// 12.7 ms, with geometry 1.38 against 1.02 and 19.8 against 11.0 (2 x 80
// triangles, 1,000,000: 11.7 against 6.9 and 13.1 against 6.9); but between 2 x
// 20,480 triangles, where the batch waits for its heaviest queries, 65,536 3.9
// against 12.2 and 3.5 against 8.9 (1,000,000: 39 against 54 and 38 against 40),
// so both only below kNarrowPairs node pairs.  With more contacts little is
// tested in vain, and whole wavefronts stay ahead (100,000 queries, 8 contacts:
// 2.3 against 3.9 ms).
constexpr int kNarrowMin = 65536;
constexpr long long kNarrowPairs = 1LL << 26;  // 2 x 4,096 triangles

// The FP64 test of a node pair the cull left unsure.
__device__ __forceinline__ bool overlap64(const QueryXf64& x, const ObbNode64* n1,
                                       const ObbNode64* n2) {
  M3 R;
#pragma unroll
  for (int i = 0; i < 9; ++i) R.m[i] = x.R[i];
  return obb_overlap64(R, v3(x.T[0], x.T[1], x.T[2]), *n1, *n2);
}

// Test of the BVTT node (b1, b2): its children, a leaf pair, or nothing.
__device__ __forceinline__ void visit_node(const CollideLaunch& L, const QueryXf32& X,
                                           const QueryPtr& P, const QueryXf64& x, int b1, int b2,
                                           OrdOutcome& r) {
  const ObbNode32 n1 = load_node32(P.n1 + b1);
  const ObbNode32 n2 = load_node32(P.n2 + b2);
  r.bv = 1;
  int c = obb_cull32(X, n1, n2);
  if (c == kCullUnsure)
    c = overlap64(x, L.meshes[X.m1].obb64 + b1, L.meshes[X.m2].obb64 + b2) ? kCullOverlap
                                                                          : kCullDisjoint;
  if (c != kCullOverlap) return;
  const int f1 = n1.first_child, f2 = n2.first_child;
  if (f1 < 0 && f2 < 0) {
    r.nout = 1;
    r.o0 = ord_pack(kOrdLeaf, -(f1 + 1), -(f2 + 1));
  } else {
    r.nout = 2;
    if ((f2 < 0) || (f1 >= 0 && first_larger(n1, n2, P.s1 + b1, P.s2 + b2))) {
      r.o0 = ord_pack(kOrdNode, f1, b2);
      r.o1 = ord_pack(kOrdNode, f1 + 1, b2);
    } else {
      r.o0 = ord_pack(kOrdNode, b1, f2);
      r.o1 = ord_pack(kOrdNode, b1, f2 + 1);
    }
  }
}

struct TriPair {
  V3 P[3], Q[3];  // each in its own mesh's frame
};

__device__ __forceinline__ TriPair load_tris(const QueryXf64& x, int t1, int t2) {
  const double* p = x.tv1 + kTriVertsStride * static_cast<size_t>(t1);
  const double* q = x.tv2 + kTriVertsStride * static_cast<size_t>(t2);
  TriPair t;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    t.P[k] = v3(p[3 * k], p[3 * k + 1], p[3 * k + 2]);
    t.Q[k] = v3(q[3 * k], q[3 * k + 1], q[3 * k + 2]);
  }
  return t;
}

// The pair's contacts (mesh_collision_traversal_node-inl.h:578-598): 0-2
// points in mesh 1's frame, with one normal and depth.
__device__ __forceinline__ unsigned tri_points(const QueryXf64& x, const M3& R, const TriPair& t,
                                               V3 (&pts)[2], V3& nrm, double& depth) {
  const V3 T = v3(x.T[0], x.T[1], x.T[2]);
  return tri_contact64(t.P[0], t.P[1], t.P[2], mul(R, t.Q[0]) + T, mul(R, t.Q[1]) + T,
                       mul(R, t.Q[2]) + T, pts, nrm, depth);
}

// The triangle test of a leaf pair: -1 for no intersection, else its contacts
// (one without contact geometry).
template <bool kContact>
__device__ __forceinline__ int leaf_contacts(const QueryXf64& x, int t1, int t2) {
  const TriPair t = load_tris(x, t1, t2);
  M3 R;
#pragma unroll
  for (int i = 0; i < 9; ++i) R.m[i] = x.R[i];
  if (!tri_intersect64(t.P[0], t.P[1], t.P[2], t.Q[0], t.Q[1], t.Q[2], R,
                       v3(x.T[0], x.T[1], x.T[2])))
    return -1;
  if constexpr (kContact) {
    V3 pts[2], nrm;
    double depth;
    return static_cast<int>(tri_points(x, R, t, pts, nrm, depth));
  }
  return 1;
}

// Records of a committed hit: slots first .. first + take - 1.
template <bool kContact>
__device__ __forceinline__ void write_records(const CollideLaunch& L, const QueryXf64& x, int q,
                                           int t1, int t2, long long first, int take) {
  V3 pts[2], nrm;
  double depth = 0;
  if constexpr (kContact) {
    M3 R;
#pragma unroll
    for (int i = 0; i < 9; ++i) R.m[i] = x.R[i];
    tri_points(x, R, load_tris(x, t1, t2), pts, nrm, depth);
  }
  const double* w = L.tf1 + 12 * static_cast<size_t>(q);
  for (int i = 0; i < take; ++i) {
    const long long slot = first + i;
    if (slot >= L.pair_capacity) {
      if (L.pairs) atomicOr(L.status, kStatusPairOverflow);  // no buffer: counts only
      continue;
    }
    L.pairs[3 * slot] = q;
    L.pairs[3 * slot + 1] = t1;
    L.pairs[3 * slot + 2] = t2;
    if constexpr (kContact) {
      const V3 p = i == 0 ? pts[0] : pts[1];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const V3 rowk = v3(w[3 * k], w[3 * k + 1], w[3 * k + 2]);
        L.contact_pos[3 * slot + k] = dot(rowk, p) + w[9 + k];
        L.contact_normal[3 * slot + k] = dot(rowk, nrm);
      }
      L.contact_depth[slot] = depth;
    }
  }
}

// Statistics: none, summed in 32 bits per list entry, and the same where the
// entries' sums could outgrow them (ord_audit).
enum : int { kNoCounts = 0, kCounts32 = 1, kAuditedCounts = 2 };

template <int G, bool kStats, bool kContact>
struct OrderedWave {
  static constexpr int kGroups = kWave / G;
  OrderedList<list_cap<G>(), kStats> list[kGroups];
  QueryXf64 x64[kGroups];
  QueryXf32 x32[kGroups];
  QueryPtr ptr[kGroups];
};

// One wavefront per block, one query per group.  leaf_min: gathered leaf
// pairs of the wavefront that start their triangle tests (a group with
// nothing else to test starts them too).  kSome: queries of L.lanes_max node
// pairs at most (and those with bad ids) are left to launch_collide_lanes; a
// wavefront looks through `chunk` queries at a time for the others.  (With
// statistics the lists of four quarters leave LDS for three wavefronts per
// SIMD.)
template <int G, int kCounts, bool kContact, bool kSome>
__global__ void __launch_bounds__(kWave, G == 16 && kCounts != kNoCounts ? 3 : 4)
    collide_ordered(CollideLaunch L, int margin, int leaf_min, int chunk) {
  constexpr int kCap = list_cap<G>();
  constexpr bool kStats = kCounts != kNoCounts;
  __shared__ OrderedWave<G, kStats, kContact> W;
  const LaneGroup<G> g;
  const int gi = g.first / G;
  OrderedList<kCap, kStats>& S = W.list[gi];
  const QueryXf64& x = W.x64[gi];
  int q = -1;  // the group's query; -2: none left
  unsigned next = blockIdx.x * (kSome ? chunk : kWave / G) + (kSome ? 0 : gi);
  unsigned from = 0;            // kSome: the chunk looked through
  unsigned long long todo = 0;  // and its queries left
  OrdTotals T;
  while (true) {
    // groups without a query take the next one
    const unsigned long long need = __ballot(g.lane == 0 && q == -1);
    if (need != 0) {
      if constexpr (kSome) {
        while (todo == 0 && next < static_cast<unsigned>(L.num_queries)) {
          from = next;
          next += gridDim.x * chunk;
          const unsigned c = from + __lane_id();
          bool heavy = static_cast<int>(__lane_id()) < chunk &&
                       c < static_cast<unsigned>(L.num_queries);
          if (heavy) {
            const int32_t* qm = L.query_meshes + 2 * static_cast<size_t>(c);
            heavy = obbrss_query_ok(L.meshes, L.num_meshes, qm[0], qm[1]) &&
                    node_pairs(L.meshes[qm[0]], L.meshes[qm[1]]) > L.lanes_max;
          }
          todo = __ballot(heavy);
        }
      }
      if (q == -1) {
        if constexpr (kSome) {
          unsigned long long m = todo;
          for (int k = __popcll(need & ((1ULL << g.first) - 1ULL)); k > 0; --k) m &= m - 1;
          q = m != 0 ? static_cast<int>(from) + __ffsll(static_cast<long long>(m)) - 1
                     : (next < static_cast<unsigned>(L.num_queries) ? -1 : -2);
        } else {
          q = next < static_cast<unsigned>(L.num_queries) ? static_cast<int>(next) : -2;
          next += gridDim.x * (kWave / G);
        }
        if (q >= 0) {
          const int32_t* qm = L.query_meshes + 2 * static_cast<size_t>(q);
          const int i1 = qm[0], i2 = qm[1];
          if (!obbrss_query_ok(L.meshes, L.num_meshes, i1, i2)) {
            if (g.lane == 0) {
              L.counts[q] = 0;
              if (L.bv_tests) L.bv_tests[q] = 0;
              if (L.leaf_tests) L.leaf_tests[q] = 0;
              atomicOr(L.status, kStatusBadQuery);
            }
            q = -1;
          } else {
            const MeshDev& m1 = L.meshes[i1];
            const MeshDev& m2 = L.meshes[i2];
            QueryXf64 y;
            rel_pose64(L.tf1 + 12 * static_cast<size_t>(q), L.tf2 + 12 * static_cast<size_t>(q),
                       y.R, y.T);
            y.tv1 = m1.tri_verts;
            y.tv2 = m2.tri_verts;
            QueryXf32 X;
            make_xf32_checked(y.R, y.T, m1.cmax, m2.cmax, X);
            X.m1 = i1;
            X.m2 = i2;
            X.valid = 1;
            if (g.lane == 0) {
              W.x64[gi] = y;
              W.x32[gi] = X;
              W.ptr[gi] = QueryPtr{m1.obb32, m2.obb32, m1.size64, m2.size64};
            }
            T = ord_begin(g, S, L.carry_max);
          }
        }
      }
      if constexpr (kSome)
        for (int k = __popcll(need); k > 0 && todo != 0; --k) todo &= todo - 1;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    if (__ballot(q != -2) == 0) break;
    // the window: lane k holds the list's entry k from the top
    int n = q >= 0 ? ord_window<G, kCap>(T.sp, margin) : 0;
    if constexpr (kCounts == kAuditedCounts)
      if (__ballot(--T.audit_in < 0) != 0) ord_audit(g, S, T, L.carry_max, n);
    const bool on = g.lane < n;
    unsigned long long e = 0;
    uint2 acc = make_uint2(0u, 0u);
    if (on) {
      e = S.e[T.sp - 1 - g.lane];
      if constexpr (kStats) acc = S.acc[T.sp - 1 - g.lane];
    }
    const int kind = ord_kind(e);
    const bool node = on && kind == kOrdNode, leaf = on && kind == kOrdLeaf;
    OrdOutcome r;
    if (on && kind >= kOrdHit) {
      r.nout = 1;
      r.o0 = e;
      r.hit = true;
      r.n = kind - kOrdHit;
    }
    const unsigned long long lm = __ballot(leaf);
    bool test_leaves = false;
    if (lm != 0) {
      // groups with leaf pairs and no node to test wait for nothing else
      const bool stuck = g.part(lm) != 0 && g.ballot(node) == 0;
      test_leaves = __popcll(lm) >= leaf_min || __ballot(stuck) != 0;
    }
    if (node) {
      visit_node(L, W.x32[gi], W.ptr[gi], x, ord_a(e), ord_b(e), r);
    } else if (leaf) {
      if (test_leaves) {
        r.leaf = 1;
        const int c = leaf_contacts<kContact>(x, ord_a(e), ord_b(e));
        if (c >= 0) {
          r.nout = 1;
          r.hit = true;
          r.n = c;
          r.o0 = ord_pack(kOrdHit + c, ord_a(e), ord_b(e));
        }
      } else {
        r.nout = 1;
        r.o0 = e;
      }
    }
    ord_settle<G, kCap, kStats>(g, S, T, r, acc, n, L.cap, [&](bool mine, int take, int before,
                                                               int total) {
      unsigned long long b = static_cast<unsigned>(T.count);  // a single query's own records
      if (L.num_pairs && g.lane == 0 && total > 0)
        b = atomicAdd(reinterpret_cast<unsigned long long*>(L.num_pairs),
                      static_cast<unsigned long long>(total));
      b = (static_cast<unsigned long long>(g.at(static_cast<unsigned>(b >> 32), 0)) << 32) |
          g.at(static_cast<unsigned>(b), 0);
      if (mine && take > 0)
        write_records<kContact>(L, x, q, ord_a(r.o0), ord_b(r.o0),
                                static_cast<long long>(b) + before, take);
    });
    if (q >= 0 && T.sp == 0) {
      if (g.lane == 0) {
        L.counts[q] = T.count;
        if constexpr (kStats) {
          if (L.bv_tests) L.bv_tests[q] = S.total.x;
          if (L.leaf_tests) L.leaf_tests[q] = S.total.y;
        }
      }
      q = -1;
    }
  }
}

}  // namespace

// Where a lane per query is the faster form: queries too light to fill a
// wavefront's steps, in batches large enough to fill the chip's lanes.
// Measured (lanes / groups): two triangles, 1,000 queries 29 / 33 us and
// 1,000,000 0.23 / 1.64 ms; a triangle and a box of 12, 16,000 queries to the
// first contact 160 / 124 us, 65,536 184 / 227, 1,000,000 to 8 contacts 2.4 /
// 5.1 ms; two boxes to the first contact 65,536 0.41 / 0.39, 250,000 1.1 / 1.3
// and 1,000,000 3.4 / 5.0 ms, to 8 contacts 12.6 / 10.4; two meshes of 20
// triangles to the first contact, 1,000,000 6.2 / 5.8.
long long collide_lanes_max(int num_queries, int cap, size_t nodes_min, size_t nodes_max) {
  const long long limit =
      num_queries >= 131072 && cap == 1
          ? 1024
          : (num_queries >= 32768 ? 32 : (num_queries >= 512 ? 1 : 0));
  return lanes_within(limit, nodes_min, nodes_max);
}

hipError_t launch_collide_ordered(const CollideLaunch& L, int stack_need, hipStream_t s) {
  if (L.num_queries <= 0) return hipSuccess;
  if (L.lanes_max > 0) {
    const hipError_t e = launch_collide_lanes(L, stack_need, s);
    if (e != hipSuccess || L.lanes_max == kAllLanes) return e;
  }
  const int margin = stack_need + 2;
  // (statistics that fit 32 bits by the meshes' sizes need no audits, which
  // take 1 % of a single call)
  const int counts = !(L.bv_tests || L.leaf_tests)
                         ? kNoCounts
                         : (L.node_pairs_max <= static_cast<long long>(L.carry_max) ? kCounts32
                                                                                     : kAuditedCounts);
  // (a quarter's list must hold a tree path and a step)
  const bool narrow = L.num_queries >= kNarrowMin && L.cap == 1 && margin + 16 <= list_cap<16>() &&
                      ((counts == kNoCounts && !L.contact) || L.node_pairs_max <= kNarrowPairs);
  const int G = narrow ? 16 : kWave;
  auto pick = [&](auto g, auto some) {
    constexpr int kG = decltype(g)::value;
    constexpr bool kSome = decltype(some)::value;
    if (counts == kNoCounts)
      return L.contact ? collide_ordered<kG, kNoCounts, true, kSome>
                       : collide_ordered<kG, kNoCounts, false, kSome>;
    if constexpr (!kSome)
      if (counts == kCounts32)
        return L.contact ? collide_ordered<kG, kCounts32, true, kSome>
                         : collide_ordered<kG, kCounts32, false, kSome>;
    return L.contact ? collide_ordered<kG, kAuditedCounts, true, kSome>
                     : collide_ordered<kG, kAuditedCounts, false, kSome>;
  };
  const std::integral_constant<int, 16> quarter;
  const std::integral_constant<int, 64> whole;
  const std::true_type some;
  const std::false_type all;
  auto kernel = L.lanes_max > 0 ? (narrow ? pick(quarter, some) : pick(whole, some))
                                : (narrow ? pick(quarter, all) : pick(whole, all));
  // A wavefront's queries to look through: few, as it answers its heavy ones one
  // after the other (a box against 20,480 triangles with statistics, 250,000
  // queries: 5.0 ms in 8,192 parts, 4.1 in 65,536, 4.0 where no query is light)
  const int chunk =
      L.lanes_max > 0 ? std::min(std::max(L.num_queries / 131072, kWave / G), kWave) : kWave / G;
  kernel<<<group_blocks((L.num_queries + chunk - 1LL) / chunk), kWave, 0, s>>>(
      L, margin, narrow ? 8 : 16, chunk);
  return hipGetLastError();
}

}  // namespace fclx
