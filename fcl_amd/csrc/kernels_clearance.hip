// distance() in the reference's order by one wavefront per query: the
// single-query call, and batches whose merged BVs make the answer depend on
// the visit order.
//
// distanceRecurse (traversal_recurse-inl.h:257-316) computes the two child
// bounds of a node, visits the nearer child and then the other one, each only
// if its bound is below the least distance found before its turn.  A
// wavefront keeps the pending nodes as a list in visit order (LDS, top
// first), computes the child bounds and triangle distances of its first 64
// entries ahead of their turns, and settles turns in order from the top:
//
//   - a node expanded ahead of its turn leaves a mark in front of its
//     children.  When the mark's turn comes, a bound below the least distance
//     counts its two tests; otherwise the mark's subtree, the entries up to
//     the next one of the mark's level or above, is removed as never visited;
//   - a triangle pair keeps its distance until its turn, and only then counts
//     and may lower the least distance;
//   - any entry whose bound is not below the least distance is removed: that
//     distance only falls.
//
// So the distance, the pair, the points and the test counts are the
// reference's.  The list stays bounded: a step adds no more entries than the
// room above a margin of one tree path, and beyond that it expands only the
// node whose turn it is, whose mark is settled at once.
//
// Bound: the chain of steps.  After the first descent few pending nodes are
// below the least distance (3-4 on average), so a step expands several levels
// below each of them.  One distance() call between 2 x 2,420 triangles (2,550
// bounds and 175 triangle distances on average): 4.2 ms on one lane, 1.5 ms a
// level at a time (200-650 steps of 3-4 us), 1.0 ms with several.
#include <hip/hip_runtime.h>

#include "device/dist64.h"
#include "device/pose64.h"
#include "kernels.h"

namespace fclx {

namespace {

constexpr int kWave = 64;
constexpr int kList = 512;  // entries; summed depth <= kMaxStack leaves room for wide steps
constexpr double kNone = 1.7976931348623157e308;  // DistanceResult::min_distance starts at max()

enum : int { kNode = 0, kLeaf = 1, kMark = 2, kDone = 3 };  // kDone: a leaf with its distance

// kind:2 | level:9 | a:26 | b:26; nodes, or triangles for kLeaf and kDone
constexpr int kIdBits = 26;
constexpr int kIdMask = (1 << kIdBits) - 1;
__device__ __forceinline__ unsigned long long entry(int kind, int level, int a, int b) {
  return (static_cast<unsigned long long>(kind) << (2 * kIdBits + 9)) |
         (static_cast<unsigned long long>(level) << (2 * kIdBits)) |
         (static_cast<unsigned long long>(a) << kIdBits) | static_cast<unsigned long long>(b);
}
__device__ __forceinline__ int kind_of(unsigned long long e) {
  return static_cast<int>(e >> (2 * kIdBits + 9));
}
__device__ __forceinline__ int level_of(unsigned long long e) {
  return static_cast<int>(e >> (2 * kIdBits)) & 511;
}
__device__ __forceinline__ int id_a(unsigned long long e) {
  return static_cast<int>(e >> kIdBits) & kIdMask;
}
__device__ __forceinline__ int id_b(unsigned long long e) { return static_cast<int>(e) & kIdMask; }

// Distance of triangles t1, t2 (model 2's moved into model 1's frame).
__device__ __forceinline__ double pair_distance(const MeshDev& m1, const MeshDev& m2, const M3& R,
                                                const V3& T, int t1, int t2, V3& P, V3& Q) {
  const double* p = m1.tri_verts + kTriVertsStride * static_cast<size_t>(t1);
  const double* q = m2.tri_verts + kTriVertsStride * static_cast<size_t>(t2);
  V3 S[3], U[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    S[k] = v3(p[3 * k], p[3 * k + 1], p[3 * k + 2]);
    U[k] = mul(R, v3(q[3 * k], q[3 * k + 1], q[3 * k + 2])) + T;
  }
  return tri_distance64(S, U, P, Q);
}

struct List {
  unsigned long long e[kList];
  double d[kList];  // the entry's bound
  double t[kList];  // kDone: the triangle distance
  int cand[kWave / 4];  // lanes of the nodes a step expands
};

__device__ __forceinline__ int first_of(unsigned long long m) {
  return m != 0 ? __ffsll(static_cast<long long>(m)) - 1 : kWave;
}

// kSome: queries of L.lanes_max node pairs at most are left to a lane each.
template <bool kSome>
__global__ void __launch_bounds__(kWave, 1) distance_ordered(DistanceLaunch L, int margin) {
  __shared__ List S;
  const int q = blockIdx.x;
  const int lane = static_cast<int>(__lane_id());
  const unsigned long long below = (1ULL << lane) - 1ULL;
  const int i1 = L.query_meshes[2 * q], i2 = L.query_meshes[2 * q + 1];
  if (!query_ok(L.meshes, L.num_meshes, i1, i2, /*need_obbrss=*/false)) {
    if (lane == 0) {
      L.distance[q] = kNone;
      if (L.ids) {
        L.ids[2 * q] = -1;
        L.ids[2 * q + 1] = -1;
      }
      if (L.bv_tests) L.bv_tests[q] = 0;
      if (L.leaf_tests) L.leaf_tests[q] = 0;
      atomicOr(L.status, kStatusBadQuery);
    }
    return;
  }
  const MeshDev& m1 = L.meshes[i1];
  const MeshDev& m2 = L.meshes[i2];
  if (kSome && node_pairs(m1, m2) <= L.lanes_max) return;
  const double* tf1 = L.tf1 + 12 * static_cast<size_t>(q);
  M3 R;
  V3 T;
  inverse_compose(tf1, L.tf2 + 12 * static_cast<size_t>(q), R, T);
  long long bv = 0, leaves = 0;
  V3 P, Q;
  // seed with triangle 0 of each model (distancePreprocessOrientedNode)
  double best = kNone;
  int best1 = -1, best2 = -1;
  {
    const double d = pair_distance(m1, m2, R, T, 0, 0, P, Q);
    if (best > d) {
      best = d;
      best1 = best2 = 0;
    }
  }
  // the root is visited whatever the seed's distance
  int sp = 1;
  int drop = -1;  // a removed mark's level while its subtree is being removed
  if (lane == 0) {
    const int f1 = m1.rss64[0].first_child, f2 = m2.rss64[0].first_child;
    S.e[0] = f1 < 0 && f2 < 0 ? entry(kLeaf, 0, -(f1 + 1), -(f2 + 1)) : entry(kNode, 0, 0, 0);
    S.d[0] = -kNone;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  while (sp > 0) {
    const int n = sp < kWave ? sp : kWave;
    const bool on = lane < n;
    const int pos = sp - 1 - lane;
    unsigned long long e = 0;
    double d = 0, t = kNone;
    if (on) {
      e = S.e[pos];
      d = S.d[pos];
      t = S.t[pos];
    }
    int kind = on ? kind_of(e) : kNode;
    bool keep = on;
    // a removed mark's subtree, at the top of the list
    if (drop >= 0) {
      const int end = first_of(__ballot(on && level_of(e) <= drop));
      if (lane < end) keep = false;
      if (end < n) drop = -1;
    }
    // entries that will not be visited
    const bool over = d >= best;
    if (keep && over && kind != kMark) keep = false;
    // the first entry left: a mark that fails its turn takes its subtree along
    const int top = first_of(__ballot(keep));
    if (top < kWave) {
      const bool fails = keep && lane == top && kind == kMark && over;
      if (__ballot(fails) != 0) {
        const int lv = __shfl(level_of(e), top);
        const int end = first_of(__ballot(on && lane > top && level_of(e) <= lv));
        if (lane >= top && lane < end) keep = false;
        if (end >= n) drop = lv;
      }
    }
    // Expansions, as many levels at once as lanes are free: a node's
    // descendants take a row of 2^(depth+1) lanes, lane i of a row (heap
    // order, 1 the node itself) the bound of one of them; which pairs they
    // are follows from the BVs' sizes alone.
    const int room = kList - margin - sp;
    const int head = first_of(__ballot(keep));  // its turn has come
    const unsigned long long nm = __ballot(keep && kind == kNode);
    const int open = __popcll(nm);
    int depth = open <= 1 ? 5 : (open <= 2 ? 4 : (open <= 4 ? 3 : (open <= 8 ? 2 : 1)));
    while (depth > 1 && (open << (depth + 1)) > room) --depth;
    const int row = 2 << depth;
    const int most = room / row < kWave / row ? room / row : kWave / row;
    const bool expand = keep && kind == kNode &&
                        (most > 0 ? __popcll(nm & below) < most : lane == head);
    const unsigned long long em = __ballot(expand);
    const int nexp = __popcll(em);
    const int mine = lane / row, heap = lane & (row - 1);  // this lane's row and place in it
    unsigned long long child = 0;  // the lane's descendant, its bound and place in visit order
    double child_d = 0;
    bool alive = false;
    int place = 0, from = 0;
    int grown = 0;  // entries the lane's node leaves below itself
    if (nexp > 0) {
      if (expand) S.cand[__popcll(em & below)] = lane;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      from = S.cand[mine < nexp ? mine : 0];
      const unsigned long long pe = __shfl(e, from);
      const int levels = heap > 0 ? 31 - __clz(heap) : 0;
      alive = mine < nexp && heap > 0;
      if (alive) {
        int b1 = id_a(pe), b2 = id_b(pe);
        int f1 = m1.rss64[b1].first_child, f2 = m2.rss64[b2].first_child;
        for (int k = levels - 1; k >= 0; --k) {
          if (f1 < 0 && f2 < 0) {  // a leaf pair has no children
            alive = false;
            break;
          }
          const int side = (heap >> k) & 1;
          if ((f2 < 0) || (f1 >= 0 && (m1.size64[b1] > m2.size64[b2]))) {
            b1 = f1 + side;
            f1 = m1.rss64[b1].first_child;
          } else {
            b2 = f2 + side;
            f2 = m2.rss64[b2].first_child;
          }
        }
        if (alive && heap > 1) {
          const int lv = level_of(pe) + levels;
          child = f1 < 0 && f2 < 0 ? entry(kLeaf, lv, -(f1 + 1), -(f2 + 1))
                                   : (levels == depth ? entry(kNode, lv, b1, b2)
                                                      : entry(kMark, lv, 0, 0));
          child_d = rss_distance64(R, T, m1.rss64[b1], m2.rss64[b2]);
          alive = !(child_d >= best);
        }
      }
      // a descendant stays if its whole path does
      const int row0 = lane - heap;
      for (int k = 1; k <= depth; ++k) {
        const bool up = __shfl(alive ? 1 : 0, row0 + (heap >> 1)) != 0;
        if (levels == k) alive = alive && up;
      }
      // entries of each subtree, from the deepest level up
      int size = alive ? 1 : 0;
      for (int k = depth - 1; k >= 0; --k) {
        const int a = __shfl(size, row0 + ((2 * heap) & (row - 1)));
        const int b = __shfl(size, row0 + ((2 * heap + 1) & (row - 1)));
        if (levels == k && alive) size += a + b;
      }
      // visit order: a node before its children, the nearer child's subtree
      // (the first on ties) before the other's
      const double other_d = __shfl_xor(child_d, 1);
      const bool far = (heap & 1) != 0 ? !(child_d < other_d) : other_d < child_d;
      const int other_size = __shfl_xor(size, 1);
      for (int k = 1; k <= depth; ++k) {
        const int up = __shfl(place, row0 + (heap >> 1));
        if (levels == k) place = up + 1 + (far ? other_size : 0);
      }
      const int total = __shfl(size, (__popcll(em & below) * row + 1) & (kWave - 1));
      grown = expand ? total - 1 : 0;
    }
    // triangle distances: when the next turn is one, or many have gathered
    const bool leaf = keep && kind == kLeaf;
    const unsigned long long lm = __ballot(leaf);
    if (lm != 0 && (nexp == 0 || __popcll(lm) >= 16 || ((lm >> head) & 1) != 0)) {
      if (leaf) {
        t = pair_distance(m1, m2, R, T, id_a(e), id_b(e), P, Q);
        e = entry(kDone, level_of(e), id_a(e), id_b(e));
        kind = kDone;
      }
    }
    // turns, from the top: marks and pairs with their distance, each against
    // the least distance before it; up to the first other entry, whose mark
    // is settled too if it was expanded
    const bool settled = keep && (kind == kMark || kind == kDone);
    const int stop = first_of(__ballot(keep && !settled));
    const double own = settled && kind == kDone && lane < stop && t < best ? t : best;
    double low = own;  // least distance up to and with this lane
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
      const double o = __shfl_up(low, s);
      if (lane >= s && o < low) low = o;
    }
    double before = __shfl_up(low, 1);
    if (lane == 0) before = best;
    const int bad = first_of(__ballot(settled && lane < stop && d >= before));
    const int end = bad < stop ? bad : stop;  // lanes below have had their turns
    const bool turn = settled && lane < end;
    bv += 2 * __popcll(__ballot(turn && kind == kMark));
    leaves += __popcll(__ballot(turn && kind == kDone));
    if (__ballot(turn && kind == kDone) != 0) {
      const double now = __shfl(low, end - 1);
      if (now < best) {
        const int w = first_of(__ballot(turn && kind == kDone && t == now));
        best1 = __shfl(id_a(e), w);
        best2 = __shfl(id_b(e), w);
        best = now;
      }
    }
    // the expanded node right after the settled turns: its turn too, if its
    // bound still is below the least distance
    const bool turn_now = expand && lane == end && !(d >= best);
    bv += 2 * __popcll(__ballot(turn_now));
    // back into the list, in visit order
    const int nout = !keep || turn ? 0 : grown + (turn_now ? 0 : 1);
    int sum = nout;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
      const int o = __shfl_up(sum, s);
      if (lane >= s) sum += o;
    }
    sp = sp - n + __shfl(sum, kWave - 1);
    const int at = sp - 1 - (sum - nout);
    if (nout > grown) {
      S.e[at] = expand ? entry(kMark, level_of(e), 0, 0) : e;
      S.d[at] = d;
      S.t[at] = t;
    }
    if (nexp > 0) {
      const int below_node = __shfl(at - (nout > grown ? 1 : 0), from);
      if (alive && heap > 1) {
        S.e[below_node - (place - 1)] = child;
        S.d[below_node - (place - 1)] = child_d;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  if (L.points && best1 >= 0) (void)pair_distance(m1, m2, R, T, best1, best2, P, Q);
  if (lane == 0) {
    L.distance[q] = best;
    if (L.ids) {
      L.ids[2 * q] = best1;
      L.ids[2 * q + 1] = best2;
    }
    if (L.points) {
      // nearest points back to the world frame through tf1
      M3 R1;
      V3 t1;
      load_pose(tf1, R1, t1);
      if (best1 < 0) P = Q = v3(0, 0, 0);
      const V3 wp = mul(R1, P) + t1, wq = mul(R1, Q) + t1;
      double* o = L.points + 6 * static_cast<size_t>(q);
      o[0] = wp.x;
      o[1] = wp.y;
      o[2] = wp.z;
      o[3] = wq.x;
      o[4] = wq.y;
      o[5] = wq.z;
    }
    if (L.bv_tests) L.bv_tests[q] = bv;
    if (L.leaf_tests) L.leaf_tests[q] = leaves;
  }
}

}  // namespace

bool distance_ordered_takes(size_t max_nodes) { return max_nodes <= (size_t(1) << kIdBits); }

// Where a lane per query is the faster form (for the queries whose chains a
// batch is large enough to hide).  Lanes / wavefronts, measured: two triangles,
// 2,000 queries 51 / 52 us and 1,000,000 0.32 / 9.2 ms; a triangle and a box
// of 12, 32,768 queries 0.56 / 0.54; two boxes 65,536 3.9 / 3.5 and 131,072
// 4.5 / 6.9; 2 x 20 triangles 65,536 5.4 / 6.1; 2 x 80, 131,072 30 / 39; 320 and
// 80, 250,000 104 / 117; 2 x 320, 250,000 194 / 189 and 1,000,000 676 / 749; 2 x
// 2,420, 250,000 1,518 / 1,432 ms.
long long distance_lanes_max(int num_queries, size_t nodes_min, size_t nodes_max) {
  long long limit = 0;
  if (num_queries >= 2048) limit = 1;
  if (num_queries >= 36864) limit = 64;
  if (num_queries >= 65536) limit = 2048;
  if (num_queries >= 98304) limit = 32768;
  if (num_queries >= 196608) limit = 131072;
  if (num_queries >= 600000) limit = 524288;
  return lanes_within(limit, nodes_min, nodes_max);
}

hipError_t launch_distance_ordered(const DistanceLaunch& L, int stack_need, hipStream_t s) {
  if (L.lanes_max > 0) {
    const hipError_t e = launch_distance_plain(L, stack_need, s);
    if (e != hipSuccess || L.lanes_max == kAllLanes) return e;
  }
  auto kernel = L.lanes_max > 0 ? distance_ordered<true> : distance_ordered<false>;
  // HIP refuses a launch of 2^32 threads: larger batches in parts (a loop in
  // the kernel took 2 % of a single call)
  constexpr int kPart = 1 << 25;
  DistanceLaunch P = L;
  for (int left = L.num_queries; left > 0; left -= kPart) {
    P.num_queries = left < kPart ? left : kPart;
    kernel<<<static_cast<unsigned>(P.num_queries), kWave, 0, s>>>(P, stack_need + 2);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    P.query_meshes += 2 * static_cast<size_t>(kPart);
    P.tf1 += 12 * static_cast<size_t>(kPart);
    P.tf2 += 12 * static_cast<size_t>(kPart);
    P.distance += kPart;
    if (P.points) P.points += 6 * static_cast<size_t>(kPart);
    if (P.ids) P.ids += 2 * static_cast<size_t>(kPart);
    if (P.bv_tests) P.bv_tests += kPart;
    if (P.leaf_tests) P.leaf_tests += kPart;
  }
  return hipSuccess;
}

}  // namespace fclx
