// Wavefront-wide mesh distance (fclx_distance_batch with FCLX_ENGINE_FAST).
//
// distanceRecurse (traversal_recurse-inl.h:257-316) visits the BVTT depth
// first, the child of smaller RSS lower bound first, and prunes a pair
// whose bound is not below the best distance so far; the first pair that
// reaches the minimum is reported (DistanceResult::update keeps it on ties,
// distance_result-inl.h:84-105).  Here a wavefront keeps kSlots queries in
// flight, each with a LIFO stack in device memory, and a step computes up
// to 64 bounds across them (an even share of 32 tasks per query, more for
// deeper stacks), so each query descends nearly depth first while the lanes
// stay busy.  Leaf pairs are queued and their FP64 triangle distances taken
// 64 at a time.
//
// Every task carries its path from the root as a key: at depth k, bit 63-k
// is 0 for the child the reference visits first and 1 for the other, so the
// reference's visit order is the order of the keys.  A query's best is the
// smallest (distance, key) found, and a task is pruned when its bound is
// above the best distance, or equal to it with a key above the best key
// (all pairs of its subtree come later in the reference's order).  Hence
// the minimum and the pair reported are the reference's whatever the order
// of the work (prunes() says what rounding asks for); the nearest points are
// those of that pair, recomputed when the query is done.
//
// Bounds are first FP32 intervals around the FP64 ones (device/rss32.h; the
// dist_fp32_cull tunable, on by default).  Where the intervals decide what the
// FP64 bounds would (each child pruned or kept, and which is nearer when both
// stay), a child goes on the stack with its interval's lower end, so later
// pruning stays safe.  When one child is left the key bit of its level is left
// 0: the other's subtree holds no pair within the best distance, so no
// comparison the bit could decide is ever made.  Where they do not (0.3 % of
// the tasks on 20,480-triangle meshes), the task goes to a queue whose FP64
// bounds (the reference's rectDistance on the 128-B FP64 nodes) are taken 64
// at a time and decide exactly as the FP64 form does; the task's two stack
// entries are reserved when it is queued (in lane order, where its children
// would have gone) and the slot takes no tasks until they are filled, so the
// stack keeps its depth-first shape and bound.
//
// Bound: latency (a wavefront waits 54 % of its cycles, at two wavefronts per
// SIMD, which is what triangle distance's registers allow).  A step's chain is the
// tasks off the stacks, their children's nodes, the bounds and the children
// onto the stacks.  So a task names its children rather than its own nodes
// (one load less in the chain), its two children have a lane each, and wavefronts
// share out a small batch one query at a time.  The FP64 form's case
// analysis made a step 14,000 cycles of divergent edge tests.  10,000 queries
// of 20,480-triangle meshes 15.5 -> 9.5 ms, 5,000 11.3 -> 5.3, 2,000 9.7 ->
// 3.2, 64 7.3 -> 2.3; of 2,420 triangles 10,000 5.4 -> 2.9.
// num_bv_tests counts this engine's bounds (FP32 and FP64 alike),
// num_leaf_tests its triangle distances.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device/pose64.h"
#include "device/rss32.h"
#include "kernels.h"

namespace fclx {
namespace {

constexpr int kDWave = 64;
constexpr int kDTasks = 32;  // tasks per step: a lane for each child
constexpr int kDBlock = 256;
constexpr int kDWaves = kDBlock / kDWave;
constexpr int kDQueue = 128;
constexpr int kDSlotCap = 1024;  // stack entries per query slot (at least)

// A task names its pair's children, so that expanding it starts with their
// loads: depth:6 | split:2 | x:21 | y:21; bound; path key.  kFirst: the first
// mesh's node is split, x is its first child and y the second mesh's node;
// kSecond the other way round; kLeaf: the two leaves.
struct DTask {
  unsigned long long t;
  double d;
  unsigned long long key;
};
enum Split : int { kLeaf = 0, kFirst = 1, kSecond = 2, kNoTask = 3 };
__device__ __forceinline__ unsigned long long dpack(int split, int x, int y, int depth) {
  return (static_cast<unsigned long long>(depth) << 44) |
         (static_cast<unsigned long long>(split) << 42) |
         (static_cast<unsigned long long>(x) << 21) | static_cast<unsigned long long>(y);
}
// the task of nodes b1, b2 with first children f1, f2 (negative: a leaf) and
// sizes s1, s2 (firstOverSecond, traversal_node_bvhs-inl.h)
__device__ __forceinline__ unsigned long long dnode(int b1, int f1, double s1, int b2, int f2,
                                                    double s2, int depth) {
  if (f1 < 0 && f2 < 0) return dpack(kLeaf, b1, b2, depth);
  return (f2 < 0 || (f1 >= 0 && s1 > s2)) ? dpack(kFirst, f1, b2, depth)
                                          : dpack(kSecond, b1, f2, depth);
}
// leaf queue entry: gen:17 | slot:5 | node1:21 | node2:21 (and the key beside it);
// an FP64-bound queue entry packs its task's x, y the same way
constexpr int kDSlotBits = 5;
constexpr int kDGenMask = (1 << (22 - kDSlotBits)) - 1;
__device__ __forceinline__ unsigned long long lpack(int tag, int i1, int i2) {
  return (static_cast<unsigned long long>(tag) << 42) |
         (static_cast<unsigned long long>(i1) << 21) | static_cast<unsigned long long>(i2);
}

// What a step reads of a slot, in 16-B words.
struct alignas(16) DistSlot {
  float pose[13];  // the slot's relative pose in float, then the bound's margin term
  int pad[3];
  const RssNode32* rss1f;
  const RssNode32* rss2f;
  const double* size1;
  const double* size2;
};

template <int kSlots>
struct DistWave {
  double pose[12][kSlots];  // relative pose R (9), T (3) of each slot, chunk-major
  DistSlot at[kSlots];
  const RssNode64* rss1[kSlots];
  const RssNode64* rss2[kSlots];
  int mesh1[kSlots], mesh2[kSlots];
  int sp[kSlots], pend[kSlots], gen[kSlots];
  int upend[kSlots];  // the slot's tasks queued for FP64 bounds (the slot takes no
                      // tasks meanwhile: their children's entries are reserved)
  double best_d[kSlots];
  unsigned long long best_key[kSlots];
  int best1[kSlots], best2[kSlots];
  long long nbv[kSlots], nleaf[kSlots];
  unsigned long long lq[kDQueue];
  unsigned long long lk[kDQueue];
  // tasks that the FP32 bounds leave open: (gen, slot, x, y), the task's key
  // and its split and depth
  unsigned long long uq[kDQueue];
  unsigned long long uk[kDQueue];
  int upos[kDQueue];  // the two stack entries reserved for the children
  unsigned char ud[kDQueue];
  // a leaf step's results, for the slots to pick their minimum
  double cd[kDWave];
  unsigned long long ck[kDWave];
  int ci1[kDWave], ci2[kDWave];
  signed char cslot[kDWave];
};

// Whether a bound prunes a task, given the best (distance, key) found: as in
// the reference where the best comes before the task.  A task that comes
// before it met a larger best there, so only a bound that is above the best
// by more than rounding prunes it: pairs around a shared vertex or edge often
// have one distance to the last bit, and bounds a last bit above it.
__device__ __forceinline__ bool prunes(double d, unsigned long long key, double bd,
                                       unsigned long long bk) {
  return key > bk ? d >= bd : d > bd * (1.0 + 1e-12);
}

template <int n>
__device__ __forceinline__ int dscan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
  if (n > 2) v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
  if (n > 4) v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
  if (n > 8) v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
  return v;
}

__device__ __forceinline__ unsigned long long dbelow() {
  return (1ULL << __lane_id()) - 1ULL;
}

template <int kSlots>
__device__ __forceinline__ void slot_pose(const DistWave<kSlots>& W, int s, M3& R, V3& T) {
#pragma unroll
  for (int i = 0; i < 9; ++i) R.m[i] = W.pose[i][s];
  T = v3(W.pose[9][s], W.pose[10][s], W.pose[11][s]);
}

// FP64 distance of triangle id1 of mesh m1 and triangle id2 of mesh m2 moved
// into m1's frame (meshDistanceOrientedNodeLeafTesting, as the plain kernel)
__device__ __forceinline__ double tri_pair(const MeshDev& m1, const MeshDev& m2, const M3& R,
                                           const V3& T, int id1, int id2, V3& P, V3& Q) {
  const int32_t* t1 = m1.tris + 3 * static_cast<size_t>(id1);
  const int32_t* t2 = m2.tris + 3 * static_cast<size_t>(id2);
  const V3 S[3] = {vertex(m1, t1[0]), vertex(m1, t1[1]), vertex(m1, t1[2])};
  const V3 Tt[3] = {mul(R, vertex(m2, t2[0])) + T, mul(R, vertex(m2, t2[1])) + T,
                    mul(R, vertex(m2, t2[2])) + T};
  return tri_distance64(S, Tt, P, Q);
}

template <int kSlots, int kWavesPerSimd, bool kF32>
__global__ void __launch_bounds__(kDBlock, kWavesPerSimd) engine_distance_wave(DistanceLaunch L,
                                                                   unsigned long long* next_q,
                                                                   DTask* stk, int slot_cap,
                                                                   int wide_cap, int width,
                                                                   int leaf_batch, int live) {
  static_assert(kSlots <= 16 && kSlots <= (1 << kDSlotBits), "slots fit a DPP row");
  __shared__ DistWave<kSlots> waves_s[kDWaves];
  const int lane = __lane_id();
  const int wave = threadIdx.x / kDWave;
  DistWave<kSlots>& W = waves_s[wave];
  const long long gw = static_cast<long long>(blockIdx.x) * kDWaves + wave;
  DTask* const stacks = stk + gw * kSlots * static_cast<long long>(slot_cap);
  const bool slot_lane = lane < kSlots;
  DTask* const mine = stacks + static_cast<long long>(slot_lane ? lane : 0) * slot_cap;
  const int nq = L.num_queries;
  int q = -1, spv = 0;
  int nx = 0, ne = 0;
  bool exhausted = false, check = true;
  int nl = 0, nu = 0;
  if (slot_lane) W.gen[lane] = 0;

  for (;;) {
    if (check) {
      check = false;
      // finish queries with nothing left: stack empty, no leaf pair queued
      if (slot_lane && q >= 0) {
        spv = W.sp[lane];
        if (spv == 0 && W.pend[lane] == 0) {
          const MeshDev& m1 = L.meshes[W.mesh1[lane]];
          const MeshDev& m2 = L.meshes[W.mesh2[lane]];
          M3 R;
          V3 T;
          slot_pose(W, lane, R, T);
          V3 P, Q;
          (void)tri_pair(m1, m2, R, T, W.best1[lane], W.best2[lane], P, Q);
          L.distance[q] = W.best_d[lane];
          if (L.ids) {
            L.ids[2 * q] = W.best1[lane];
            L.ids[2 * q + 1] = W.best2[lane];
          }
          if (L.points) {
            M3 R1;
            V3 t1;
            load_pose(L.tf1 + 12 * static_cast<size_t>(q), R1, t1);
            const V3 wp = mul(R1, P) + t1, wq = mul(R1, Q) + t1;
            double* o = L.points + 6 * static_cast<size_t>(q);
            o[0] = wp.x; o[1] = wp.y; o[2] = wp.z;
            o[3] = wq.x; o[4] = wq.y; o[5] = wq.z;
          }
          if (L.bv_tests) L.bv_tests[q] = W.nbv[lane];
          if (L.leaf_tests) L.leaf_tests[q] = W.nleaf[lane];
          q = -1;
          spv = 0;
        }
      }
      const int tasks = __builtin_amdgcn_readlane(dscan<kSlots>(spv), kSlots - 1);
      unsigned long long freem = __ballot(lane < live && q < 0);
      if (!exhausted && freem != 0 && (__popcll(freem) >= 2 || tasks < kDTasks || live == 1)) {
        while (freem != 0) {
          if (nx == ne) {
            unsigned long long b = 0;
            if (lane == 0) b = atomicAdd(next_q, static_cast<unsigned long long>(live));
            b = __shfl(b, 0);
            if (b >= static_cast<unsigned long long>(nq)) {
              exhausted = true;
              break;
            }
            nx = static_cast<int>(b);
            ne = nq - nx < live ? nq : nx + live;
          }
          const int r = __popcll(freem & dbelow());
          const int n = __popcll(freem) < ne - nx ? __popcll(freem) : ne - nx;
          if (lane < live && q < 0 && r < n) {
            q = nx + r;
            const int i1 = L.query_meshes[2 * q], i2 = L.query_meshes[2 * q + 1];
            if (!query_ok(L.meshes, L.num_meshes, i1, i2, /*need_obbrss=*/false)) {
              L.distance[q] = 1.7976931348623157e308;
              if (L.ids) {
                L.ids[2 * q] = -1;
                L.ids[2 * q + 1] = -1;
              }
              if (L.bv_tests) L.bv_tests[q] = 0;
              if (L.leaf_tests) L.leaf_tests[q] = 0;
              atomicOr(L.status, kStatusBadQuery);
              q = -1;
            } else {
              const MeshDev& m1 = L.meshes[i1];
              const MeshDev& m2 = L.meshes[i2];
              M3 R;
              V3 T;
              inverse_compose(L.tf1 + 12 * static_cast<size_t>(q),
                              L.tf2 + 12 * static_cast<size_t>(q), R, T);
#pragma unroll
              for (int k = 0; k < 9; ++k) W.pose[k][lane] = R.m[k];
              W.pose[9][lane] = T.x;
              W.pose[10][lane] = T.y;
              W.pose[11][lane] = T.z;
#pragma unroll
              for (int k = 0; k < 9; ++k) W.at[lane].pose[k] = static_cast<float>(R.m[k]);
              W.at[lane].pose[9] = static_cast<float>(T.x);
              W.at[lane].pose[10] = static_cast<float>(T.y);
              W.at[lane].pose[11] = static_cast<float>(T.z);
              W.at[lane].pose[12] = rss_margin32(m1.rcmax, m2.rcmax, R, T);
              W.rss1[lane] = m1.rss64;
              W.rss2[lane] = m2.rss64;
              W.at[lane].rss1f = m1.rss32;
              W.at[lane].rss2f = m2.rss32;
              W.at[lane].size1 = m1.size64;
              W.at[lane].size2 = m2.size64;
              W.mesh1[lane] = i1;
              W.mesh2[lane] = i2;
              // seed: triangle 0 with triangle 0 (distancePreprocessOrientedNode)
              V3 P, Q;
              W.best_d[lane] = tri_pair(m1, m2, R, T, 0, 0, P, Q);
              W.best_key[lane] = 0;
              W.best1[lane] = 0;
              W.best2[lane] = 0;
              W.nbv[lane] = 0;
              W.nleaf[lane] = 0;
              mine[0] = DTask{dnode(0, m1.rss64[0].first_child, m1.size64[0], 0,
                                    m2.rss64[0].first_child, m2.size64[0], 0),
                              -1.0, 0};  // the root, never pruned
              W.sp[lane] = 1;
              W.pend[lane] = 0;
              W.upend[lane] = 0;
              W.gen[lane] = (W.gen[lane] + 1) & kDGenMask;
              spv = 1;
            }
          }
          nx += n;
          freem = __ballot(lane < live && q < 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      }
      if (exhausted && __ballot(slot_lane && q >= 0) == 0) break;
    }

    // tasks per slot: an even share, then the rest to deeper stacks, up to
    // `width` (all once every query is taken), one at a time near the cap.
    // A slot with tasks waiting for FP64 bounds takes none: their children
    // go on its stack first, so the slot keeps descending depth first and
    // its stack keeps the bound below.
    const int lim = wide_cap - spv > 1 ? wide_cap - spv : 1;
    const int wmax = exhausted ? kDTasks : width;
    const int cap_w = wmax < lim ? wmax : lim;
    const int avail = (slot_lane && W.upend[lane] > 0) ? 0 : spv;
    int take = avail < kDTasks / kSlots ? avail : kDTasks / kSlots;
    take = take < cap_w ? take : cap_w;
    int incl = dscan<kSlots>(take);
    int total = __builtin_amdgcn_readlane(incl, kSlots - 1);
    if (total < kDTasks) {
      const int e = (avail < cap_w ? avail : cap_w) - take;
      const int ei = dscan<kSlots>(e);
      const int room = kDTasks - total - (ei - e);
      take += room <= 0 ? 0 : (room < e ? room : e);
      incl = dscan<kSlots>(take);
      total = __builtin_amdgcn_readlane(incl, kSlots - 1);
    }
    const int excl = incl - take;

    if (nl >= leaf_batch || (total == 0 && nl > 0)) {
      // FP64 triangle distances of queued leaf pairs
      const int n = nl < kDWave ? nl : kDWave;
      nl -= n;
      int slot = -1;
      if (lane < n) {
        const unsigned long long e = W.lq[nl + lane];
        const unsigned long long key = W.lk[nl + lane];
        const int tag = static_cast<int>(e >> 42);
        int id1 = static_cast<int>((e >> 21) & 0x1FFFFF), id2 = static_cast<int>(e & 0x1FFFFF);
        const int s = tag & ((1 << kDSlotBits) - 1);
        if ((tag >> kDSlotBits) == W.gen[s]) {
          const int l1 = id1, l2 = id2;  // the leaf nodes
          id1 = -(W.at[s].rss1f[l1].first_child + 1);
          id2 = -(W.at[s].rss2f[l2].first_child + 1);
          const MeshDev& m1 = L.meshes[W.mesh1[s]];
          const MeshDev& m2 = L.meshes[W.mesh2[s]];
          M3 R;
          V3 T;
          slot_pose(W, s, R, T);
          V3 P, Q;
          const double d = tri_pair(m1, m2, R, T, id1, id2, P, Q);
          // a nearer pair that comes after the best found: its own bound,
          // which rounding can lift above its distance, may prune it
          const double bd = W.best_d[s];
          const bool counts =
              !(d < bd && key > W.best_key[s]) ||
              rss_distance64(R, T, W.rss1[s][l1], W.rss2[s][l2]) < bd;
          W.cd[lane] = d;
          W.ck[lane] = key;
          W.ci1[lane] = id1;
          W.ci2[lane] = id2;
          if (counts) slot = s;
          atomicSub(&W.pend[s], 1);
          atomicAdd(reinterpret_cast<unsigned long long*>(&W.nleaf[s]), 1ULL);
        }
      }
      W.cslot[lane] = static_cast<signed char>(slot);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (slot_lane) {
        // the slot's smallest (distance, key), found before or now
        double bd = W.best_d[lane];
        unsigned long long bk = W.best_key[lane];
        int b1 = W.best1[lane], b2 = W.best2[lane];
        for (int j = 0; j < n; ++j) {
          if (W.cslot[j] != lane) continue;
          const double d = W.cd[j];
          const unsigned long long k = W.ck[j];
          if (d < bd || (d == bd && k < bk)) {
            bd = d;
            bk = k;
            b1 = W.ci1[j];
            b2 = W.ci2[j];
          }
        }
        W.best_d[lane] = bd;
        W.best_key[lane] = bk;
        W.best1[lane] = b1;
        W.best2[lane] = b2;
      }
      check = true;
    } else if (kF32 && (nu >= kDWave / 2 || (total == 0 && nu > 0))) {
      // FP64 bounds of both children of up to 32 queued tasks, one bound per
      // lane (lanes 2j and 2j+1: task j's two children); the reference's
      // rectDistance decides their order (the key bit) and their pruning
      const int n = nu < kDWave / 2 ? nu : kDWave / 2;
      nu -= n;
      const int j = lane >> 1;
      const bool second = (lane & 1) != 0;
      int slot = 0, pos = 0;
      bool live = false;
      double dm = 0.0;
      int depth = 0;
      unsigned long long key = 0, task = 0;
      if (j < n) {
        const unsigned long long e = W.uq[nu + j];
        key = W.uk[nu + j];
        depth = W.ud[nu + j] & 63;
        pos = W.upos[nu + j];
        const int tag = static_cast<int>(e >> 42), split = W.ud[nu + j] >> 6;
        slot = tag & ((1 << kDSlotBits) - 1);
        live = (tag >> kDSlotBits) == W.gen[slot];
        if (live) {
          const int b1 = static_cast<int>((e >> 21) & 0x1FFFFF) + (second && split == kFirst);
          const int b2 = static_cast<int>(e & 0x1FFFFF) + (second && split == kSecond);
          const RssNode64& n1 = W.rss1[slot][b1];
          const RssNode64& n2 = W.rss2[slot][b2];
          task = dnode(b1, n1.first_child, W.at[slot].size1[b1], b2, n2.first_child,
                       W.at[slot].size2[b2], depth + 1);
          M3 R;
          V3 T;
          slot_pose(W, slot, R, T);
          dm = rss_distance64(R, T, n1, n2);
        }
      }
      const double dother = __shfl_xor(dm, 1);
      const unsigned long long other = __shfl_xor(task, 1);
      if (live && !second) {
        const double d1 = dm, d2 = dother;
        const double bd = W.best_d[slot];
        const unsigned long long bk = W.best_key[slot];
        const unsigned long long bit = 1ULL << (63 - depth);
        // the reference visits the nearer child first (a on ties)
        DTask near, far;
        if (d2 < d1) {
          near = DTask{other, d2, key};
          far = DTask{task, d1, key | bit};
        } else {
          near = DTask{task, d1, key};
          far = DTask{other, d2, key | bit};
        }
        const bool keep_far = !prunes(far.d, far.key, bd, bk);
        const bool keep_near = !prunes(near.d, near.key, bd, bk);
        // the reserved entries: far below near, so near comes off first; a
        // pruned child leaves an entry that is pruned when it comes off
        const DTask dead{dpack(kNoTask, 0, 0, 0), INFINITY, ~0ULL};
        if (pos + 2 <= slot_cap) {
          DTask* st = stacks + static_cast<long long>(slot) * slot_cap;
          st[pos] = keep_far ? far : dead;
          st[pos + 1] = keep_near ? near : dead;
        }
        atomicSub(&W.pend[slot], 1);
        atomicSub(&W.upend[slot], 1);
        atomicAdd(reinterpret_cast<unsigned long long*>(&W.nbv[slot]), 2ULL);
      }
      check = true;
    } else if (total > 0) {
      // bounds of the children of the tasks on top of the stacks (FP64, or
      // FP32 intervals with FP64 for the tasks they leave open)
      int slot = 0, first = 0, at = 0;
      const int j = lane >> 1;
      const bool second = (lane & 1) != 0;  // this lane's child is e, not a
      bool expand = false, leafc = false, unsure = false, keep = false, above = false;
      DTask c{0, 0, 0};
      int x = 0, y = 0, split = 0, depth = 0;
      unsigned long long ukey = 0, bk = 0;
      double bd = 0;
      float lo = 0, hi = 0;
      // the slot that task j falls to, and where its tasks start (a slot that
      // takes none has the next one's start)
      {
        const int base = spv - take;
        at = __builtin_amdgcn_readlane(base, 0);
#pragma unroll
        for (int k = 1; k < kSlots; ++k) {
          const int from = __builtin_amdgcn_readlane(excl, k);
          const int top = __builtin_amdgcn_readlane(base, k);
          if (j >= from) {
            slot = k;
            first = 2 * from;
            at = top;
          }
        }
      }
      if (j < total) {
        const DTask t = stacks[static_cast<long long>(slot) * slot_cap + at + j - first / 2];
        bd = W.best_d[slot];
        bk = W.best_key[slot];
        depth = static_cast<int>(t.t >> 44);
        split = static_cast<int>(t.t >> 42) & 3;
        const bool pruned = prunes(t.d, t.key, bd, bk) || split == kNoTask;
        x = static_cast<int>((t.t >> 21) & 0x1FFFFF);
        y = static_cast<int>(t.t & 0x1FFFFF);
        ukey = t.key;
        if (!pruned && split == kLeaf) {
          leafc = !second;
        } else if (!pruned) {
          expand = true;
          const int b1 = x + (second && split == kFirst), b2 = y + (second && split == kSecond);
          const DistSlot& D = W.at[slot];
          const double s1 = D.size1[b1], s2 = D.size2[b2];
          if constexpr (kF32) {
            const RssNode32& n1 = D.rss1f[b1];
            const RssNode32& n2 = D.rss2f[b2];
            c.t = dnode(b1, n1.first_child, s1, b2, n2.first_child, s2, depth + 1);
            rss_interval32(D.pose, D.pose + 9, D.pose[12], n1, n2, lo, hi);
            c.d = static_cast<double>(lo);
          } else {
            const RssNode64& n1 = W.rss1[slot][b1];
            const RssNode64& n2 = W.rss2[slot][b2];
            c.t = dnode(b1, n1.first_child, s1, b2, n2.first_child, s2, depth + 1);
            M3 R;
            V3 T;
            slot_pose(W, slot, R, T);
            c.d = rss_distance64(R, T, n1, n2);
          }
        }
      }
      // the pair's lanes see each other's bounds and agree on the children
      // that stay; above: this child goes on top of the other
      const unsigned long long bit = 1ULL << (63 - depth);
      c.key = ukey;
      if constexpr (kF32) {
        const float olo = __shfl_xor(lo, 1), ohi = __shfl_xor(hi, 1);
        if (expand) {
          // k: a child stays, as its FP64 bound would; p: it is pruned
          const bool k = static_cast<double>(hi) < bd, p = static_cast<double>(lo) > bd;
          const bool ok = static_cast<double>(ohi) < bd, op = static_cast<double>(olo) > bd;
          // (a is first where both distances are 0)
          const float la = second ? olo : lo, ha = second ? ohi : hi;
          const float le = second ? lo : olo, he = second ? hi : ohi;
          const bool a_first = ha < le || ha <= 0.0f, e_first = he < la && la > 0.0f;
          // undecided, or their order is: two stack entries are reserved for
          // their FP64 bounds in lane order, so the stack stays as the pushes
          // of the FP64 bounds would have left it
          unsure = !(k || p) || !(ok || op) || (k && ok && !a_first && !e_first);
          keep = k || unsure;
          above = k && ok && second == e_first;
          if (k && ok && !above) c.key |= bit;  // the far one, below the near
        }
      } else {
        const double od = __shfl_xor(c.d, 1);
        if (expand) {
          // the reference visits the nearer child first (a on ties)
          const bool e_first = second ? c.d < od : od < c.d;
          const bool near = second == e_first;
          const unsigned long long okey = near ? ukey | bit : ukey;
          if (!near) c.key |= bit;
          keep = !prunes(c.d, c.key, bd, bk);
          above = near && !prunes(od, okey, bd, bk);
        }
      }
      // children to the slots' stacks, in lane order
      const unsigned long long km = __ballot(keep);
      int o_stack = 0;
      if (keep) {
        const unsigned long long same = ~((1ULL << first) - 1ULL) & ((1ULL << (lane & ~1)) - 1ULL);
        o_stack = at + __popcll(km & same);
        if (!unsure && o_stack + (above ? 1 : 0) < slot_cap)
          stacks[static_cast<long long>(slot) * slot_cap + o_stack + (above ? 1 : 0)] = c;
      }
      const unsigned long long lm = __ballot(leafc);
      if (leafc) {
        const int o = nl + __popcll(lm & dbelow());
        W.lq[o] = lpack((W.gen[slot] << kDSlotBits) | slot, x, y);
        W.lk[o] = ukey;
      }
      nl += __popcll(lm);
      const unsigned long long um = __ballot(unsure && !second);
      if (unsure && !second) {
        const int o = nu + __popcll(um & dbelow());
        W.uq[o] = lpack((W.gen[slot] << kDSlotBits) | slot, x, y);
        W.uk[o] = ukey;
        W.upos[o] = o_stack;
        W.ud[o] = static_cast<unsigned char>(split << 6 | depth);
      }
      nu += __popcll(um);
      const unsigned long long em = __ballot(expand);
      bool emptied = false;
      if (slot_lane && take > 0) {
        const unsigned long long own =
            (take >= kDTasks ? ~0ULL : ((1ULL << (2 * take)) - 1ULL)) << (2 * excl);
        const int nsp = spv - take + __popcll(km & own);
        if (nsp > slot_cap) {
          atomicOr(L.status, kStatusStackOverflow);
          spv = 0;  // the query's answer is incomplete; the status says so
        } else {
          spv = nsp;
        }
        W.sp[lane] = spv;
        W.pend[lane] += __popcll((lm | um) & own);
        W.upend[lane] += __popcll(um & own);
        W.nbv[lane] += __popcll(em & own);
        emptied = spv == 0;
      }
      if (__ballot(emptied) != 0) check = true;
    } else {
      check = true;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
}

__global__ void dist_zero(unsigned long long* p) { *p = 0; }

}  // namespace

hipError_t launch_distance_wave(const DistanceLaunch& L, int stack_need, const DistanceTuning& tu,
                                hipStream_t s) {
  if (L.num_queries == 0) return hipSuccess;
  // path keys hold 63 levels of descent
  if (stack_need > 62) return launch_distance_plain(L, stack_need, s);
  int dev = 0, cus = 0;
  hipError_t e;
  if ((e = hipGetDevice(&dev)) != hipSuccess ||
      (e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) !=
          hipSuccess)
    return e;
  const int K = tu.queries_per_wave;
  const int wps = tu.waves_per_simd;
  const int width = std::min(std::max(tu.width, kDTasks / K), kDTasks);
  const int leaf_batch = tu.leaf_batch;
  const long long nw = std::max<long long>(
      1, std::min<long long>(L.num_queries, static_cast<long long>(cus) * 4 * wps));
  // queries a wavefront keeps in flight: it takes a new one as one ends, so
  // few at a time spread the heavy ones (10,000 queries by four at a time
  // took 10.3 ms, by two 9.5; 50,000 by two 33.7, by four 31.8)
  const int live = static_cast<int>(std::clamp<long long>(L.num_queries / (2 * nw), 1, K));
  const unsigned grid = static_cast<unsigned>((nw + kDWaves - 1) / kDWaves);
  // as the BOOL engine: sorted by level, at most 2 entries per level above
  // the point where steps go one task at a time
  const int slot_cap = std::max(kDSlotCap, 4 * (stack_need + 2) + 2 * kDQueue);
  const int wide_cap = slot_cap - (stack_need + 2) - 2 * kDQueue;
  DTask* stk = nullptr;
  unsigned long long* ctr = nullptr;
  if ((e = hipMallocAsync(reinterpret_cast<void**>(&stk),
                          sizeof(DTask) * static_cast<size_t>(grid) * kDWaves * K * slot_cap,
                          s)) != hipSuccess)
    return e;
  if ((e = hipMallocAsync(reinterpret_cast<void**>(&ctr), sizeof(unsigned long long), s)) !=
      hipSuccess) {
    (void)hipFreeAsync(stk, s);
    return e;
  }
  dist_zero<<<1, 1, 0, s>>>(ctr);
#define FCLX_DIST(k, w, f)                                                               \
  engine_distance_wave<k, w, f><<<grid, kDBlock, 0, s>>>(L, ctr, stk, slot_cap, wide_cap, width, \
                                                         leaf_batch, live)
  if (tu.fp32_cull) {
    if (K == 2)
      wps >= 3 ? FCLX_DIST(2, 3, true) : FCLX_DIST(2, 2, true);
    else if (K == 8)
      wps >= 3 ? FCLX_DIST(8, 3, true) : FCLX_DIST(8, 2, true);
    else
      wps >= 3 ? FCLX_DIST(4, 3, true) : FCLX_DIST(4, 2, true);
  } else {
    if (K == 2)
      wps >= 3 ? FCLX_DIST(2, 3, false) : FCLX_DIST(2, 2, false);
    else if (K == 8)
      wps >= 3 ? FCLX_DIST(8, 3, false) : FCLX_DIST(8, 2, false);
    else
      wps >= 3 ? FCLX_DIST(4, 3, false) : FCLX_DIST(4, 2, false);
  }
#undef FCLX_DIST
  e = hipGetLastError();
  (void)hipFreeAsync(ctr, s);
  (void)hipFreeAsync(stk, s);
  return e;
}

}  // namespace fclx
