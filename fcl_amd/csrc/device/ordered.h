// Depth-first traversal in the reference's order by a group of lanes.
//
// The reference's recursion visits one BVTT node after the other; which
// contacts a capped query returns and its num_bv_tests / num_leaf_tests
// follow from that order.  A group (16 or 64 lanes of one wavefront)
// keeps the recursion's pending work as a list in visit order -- the LDS
// stack, its top the next node -- and tests the first entries of the list
// all at once, one per lane.  Tested entries are replaced in place: by
// nothing (disjoint), by their two children, by a leaf pair waiting for its
// triangle test, or by a hit.  So the list stays in visit order whatever was
// tested ahead of its turn, and a hit counts once everything before it is
// gone.  When hits reach num_max_contacts, what follows the last of them in
// the list is dropped, as the recursion would never have come to it.
//
// Test counts: every entry carries the tests already done on nodes that lie
// before it in visit order and after the entry before it.  An entry that
// vanishes hands its tests to the next one; dropped entries take theirs
// along.  The sums are exactly the recursion's counts.  Entries carry 32
// bits, totals 64: before the list can carry carry_max tests (2^31 unless set
// lower) ord_audit counts the top entry's, which lie before anything that can
// still be dropped, and has the group take one entry at a time while the list
// carries too many.
//
// Stack bound: a step that takes n entries grows the list by at most n.  A
// group takes no more than the room left above a margin of one tree path,
// and at least one, so beyond the margin it grows like the recursion's own
// stack: at most one entry per level.
#pragma once
#include <hip/hip_runtime.h>

namespace fclx {

template <int G>
struct LaneGroup {
  static_assert(G == 16 || G == 64, "a quarter of a wavefront or all of it");
  static constexpr unsigned long long kAll = G == 64 ? ~0ULL : (1ULL << (G & 63)) - 1ULL;
  int first;  // first lane of the group in its wavefront
  int lane;   // this lane in its group
  __device__ __forceinline__ LaneGroup() {
    const int l = __lane_id();
    lane = G == 64 ? l : l & (G - 1);
    first = G == 64 ? 0 : l - lane;
  }
  // the group's lanes with p set, bit 0 = its first lane
  __device__ __forceinline__ unsigned long long ballot(bool p) const {
    return part(__ballot(p));
  }
  __device__ __forceinline__ unsigned long long part(unsigned long long m) const {
    return G == 64 ? m : (m >> first) & kAll;
  }
  __device__ __forceinline__ unsigned long long below() const { return (1ULL << lane) - 1ULL; }
  // v of the group's lane `from`; at() with the same `from` in all lanes of
  // the group, which a whole-wavefront group reads without LDS
  __device__ __forceinline__ unsigned get(unsigned v, int from) const {
    return __shfl(v, first + from);
  }
  __device__ __forceinline__ unsigned at(unsigned v, int from) const {
    if constexpr (G == 64)
      return static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(v), from));
    else
      return __shfl(v, first + from);
  }
  // inclusive sum over the group's lanes
  __device__ __forceinline__ unsigned scan(unsigned v) const {
#pragma unroll
    for (int d = 1; d < G; d <<= 1) {
      const unsigned o = __shfl_up(v, d, G);
      if (lane >= d) v += o;
    }
    return v;
  }
};

// A list entry: kind and two 30-bit indices (a node pair, or a triangle pair
// once the BVs of a leaf pair have been found to overlap).
enum : int { kOrdNode = 0, kOrdLeaf = 1, kOrdHit = 2 };  // kOrdHit + n: n contacts (0..2)
constexpr int kOrdIndexBits = 30;
constexpr int kOrdMaxNodes = 1 << kOrdIndexBits;

__device__ __forceinline__ unsigned long long ord_pack(int kind, int a, int b) {
  return (static_cast<unsigned long long>(kind) << (2 * kOrdIndexBits)) |
         (static_cast<unsigned long long>(a) << kOrdIndexBits) |
         static_cast<unsigned long long>(b);
}
__device__ __forceinline__ int ord_kind(unsigned long long e) {
  return static_cast<int>(e >> (2 * kOrdIndexBits));
}
__device__ __forceinline__ int ord_a(unsigned long long e) {
  return static_cast<int>(e >> kOrdIndexBits) & (kOrdMaxNodes - 1);
}
__device__ __forceinline__ int ord_b(unsigned long long e) {
  return static_cast<int>(e) & (kOrdMaxNodes - 1);
}

// The list of one group (in LDS): entries and, with statistics, the tests
// each carries (BV tests and leaf tests).
template <int kCap, bool kStats>
struct OrderedList {
  unsigned long long e[kCap];
  uint2 acc[kStats ? kCap : 1];
  // The query's BV (x) and leaf (y) tests up to the last commit and behind
  // the last entry, kept by lane 0 (here rather than in registers, which the
  // kernels are short of).
  longlong2 total, tail;
};

// What a step made of this lane's entry (lanes past the step's window: none).
struct OrdOutcome {
  int nout = 0;                // entries it leaves: 0, 1 or 2
  unsigned long long o0, o1;   // in visit order
  bool hit = false;            // o0 is a hit (kOrdHit + n)
  int n = 0;                   // its contacts
  unsigned bv = 0, leaf = 0;   // tests done on it in this step
};

// State of a group's query (the same values in all its lanes).
struct OrdTotals {
  int sp = 0;
  int count = 0;     // contacts committed
  int audit_in = 0;  // steps before the next ord_audit
};

// A query's list with the root in it.
template <int G, int kCap, bool kStats>
__device__ __forceinline__ OrdTotals ord_begin(const LaneGroup<G>& g, OrderedList<kCap, kStats>& S,
                                               unsigned carry_max) {
  OrdTotals W;
  W.sp = 1;
  W.audit_in = static_cast<int>(carry_max / 128);
  if (g.lane == 0) {
    S.e[0] = ord_pack(kOrdNode, 0, 0);
    if constexpr (kStats) {
      S.acc[0] = make_uint2(0u, 0u);
      S.total = S.tail = make_longlong2(0, 0);
    }
  }
  return W;
}

// Entries the group takes from the top of its list in a step.
template <int G, int kCap>
__device__ __forceinline__ int ord_window(int sp, int margin) {
  const int room = kCap - margin - sp;
  int n = sp < G ? sp : G;
  if (n > room) n = room > 1 ? room : 1;
  return n;
}

// Before a step's window of n entries is read, once audit_in steps are over
// (adding the top's tests to the totals in each step took 3 % of a single
// call).  A list that carries less than half of carry_max goes on for as many
// full steps as cannot add the other half (64 tests each); else the step takes
// the top entry alone, whose tests reach the totals in the next one.  Either
// way no entry comes to carry more than carry_max + 64.
template <int G, int kCap>
__device__ __forceinline__ void ord_audit(const LaneGroup<G>& g, OrderedList<kCap, true>& S,
                                          OrdTotals& W, unsigned carry_max, int& n) {
  if (g.lane == 0 && n > 0) {
    const uint2 top = S.acc[W.sp - 1];
    S.total = make_longlong2(S.total.x + top.x, S.total.y + top.y);
    S.acc[W.sp - 1] = make_uint2(0u, 0u);
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  unsigned sum = 0;  // (carries below 2^32 in all)
  for (int k = g.lane; k < W.sp; k += G) sum += S.acc[k].x;
#pragma unroll
  for (int d = 1; d < G; d <<= 1) sum += __shfl_xor(sum, d);
  const bool many = sum >= carry_max / 2;
  if (many && n > 1) n = 1;
  W.audit_in = many ? 0 : static_cast<int>(carry_max / 128);
}

// Puts a step's outcomes back.  Leading hits are committed: emit(mine,
// before, take, total) is called by all lanes of the wavefront with whether
// this lane's hit is committed, how many of its contacts count, the contacts
// committed before it in this step and the group's total.  The rest of the
// window goes back in visit order, and the list ends with the hit that
// reaches the cap.  n: the window's entries (0 for a group without a query);
// acc: the tests this lane's entry carried.  W.sp = 0 afterwards: the query
// is answered.
template <int G, int kCap, bool kStats, typename Emit>
__device__ __forceinline__ void ord_settle(const LaneGroup<G>& g, OrderedList<kCap, kStats>& S,
                                           OrdTotals& W, const OrdOutcome& r, uint2 acc, int n,
                                           int cap, Emit emit) {
  int base = W.sp - n;
  const bool on = g.lane < n;
  int nout = on ? r.nout : 0;
  const bool hit = on && r.hit;
  int last = n - 1;    // last lane whose entry stays in question
  int committed = -1;  // last lane committed
  if (__ballot(hit) != 0) {
    const unsigned long long hm = g.ballot(hit);
    const unsigned own = hit ? static_cast<unsigned>(r.n) : 0u;
    const int before = static_cast<int>(g.scan(own) - own);
    const int room = cap - W.count - before;
    const unsigned long long reach = g.ballot(hit && r.n > 0 && r.n >= room);
    if (reach != 0) {
      last = __ffsll(static_cast<long long>(reach)) - 1;
      base = 0;
      if constexpr (kStats)
        if (g.lane == 0) S.tail = make_longlong2(0, 0);
      if (g.lane > last) nout = 0;
    }
    const unsigned long long open = g.ballot(nout > 0 && !hit);
    unsigned long long lm = hm;  // hits before the first open entry, up to the cap's
    if (open != 0) lm &= (open & (~open + 1ULL)) - 1ULL;
    if (reach != 0) lm &= (reach & (~reach + 1ULL)) * 2ULL - 1ULL;
    if (lm != 0) committed = 63 - __clzll(static_cast<long long>(lm));
    const bool mine = ((lm >> g.lane) & 1) != 0;
    const int take = mine ? (r.n < room ? r.n : room) : 0;
    const unsigned sum = g.at(static_cast<unsigned>(before + take), committed < 0 ? 0 : committed);
    const int total = committed < 0 ? 0 : static_cast<int>(sum);
    emit(mine, take, before, total);
    W.count += total;
    if (mine) nout = 0;
  }
  // lane 0's first entry on top
  const unsigned long long m1 = g.ballot(nout >= 1), m2 = g.ballot(nout == 2);
  const int sp = base + __popcll(m1) + __popcll(m2);
  const int at = sp - 1 - (__popcll(m1 & g.below()) + __popcll(m2 & g.below()));
  if (nout >= 1) S.e[at] = r.o0;
  if (nout == 2) S.e[at - 1] = r.o1;
  if constexpr (kStats) {
    const bool counts = on && g.lane <= last;
    const unsigned pb = g.scan(counts ? acc.x + r.bv : 0u);
    const unsigned pl = g.scan(counts ? acc.y + r.leaf : 0u);
    // an entry carries the tests since the entry or commit before it
    const unsigned long long prev = m1 & g.below();
    int from = prev != 0 ? 63 - __clzll(static_cast<long long>(prev)) : -1;
    if (committed > from) from = committed;
    const unsigned fb = g.get(pb, from < 0 ? 0 : from), fl = g.get(pl, from < 0 ? 0 : from);
    if (nout >= 1) S.acc[at] = make_uint2(pb - (from < 0 ? 0u : fb), pl - (from < 0 ? 0u : fl));
    if (nout == 2) S.acc[at - 1] = make_uint2(0u, 0u);
    // tests behind the window's last entry or commit: to the entry below
    // the window, or to the end of the list
    int end = m1 != 0 ? 63 - __clzll(static_cast<long long>(m1)) : -1;
    if (committed > end) end = committed;
    const unsigned eb = g.at(pb, end < 0 ? 0 : end), el = g.at(pl, end < 0 ? 0 : end);
    const unsigned tb = g.at(pb, G - 1) - (end < 0 ? 0u : eb);
    const unsigned tl = g.at(pl, G - 1) - (end < 0 ? 0u : el);
    const unsigned cb = g.at(pb, committed < 0 ? 0 : committed);
    const unsigned cl = g.at(pl, committed < 0 ? 0 : committed);
    if (g.lane == 0 && n > 0) {
      if (committed >= 0) S.total = make_longlong2(S.total.x + cb, S.total.y + cl);
      if (base > 0) {
        const uint2 a = S.acc[base - 1];
        S.acc[base - 1] = make_uint2(a.x + tb, a.y + tl);
      } else {
        S.tail = make_longlong2(S.tail.x + tb, S.tail.y + tl);
      }
    }
  }
  W.sp = sp;
  if (n > 0 && (sp == 0 || W.count >= cap)) {
    W.sp = 0;
    if constexpr (kStats)  // below the cap the whole tree was visited
      if (g.lane == 0 && W.count < cap)
        S.total = make_longlong2(S.total.x + S.tail.x, S.total.y + S.tail.y);
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

}  // namespace fclx
