// EPA by a group of lanes, its polytope in LDS, with the answers of shape64.h's
// one-lane form (epa-inl.h:54-396).  The lanes share a pass's arithmetic --
// the convex support's vertex scan, which faces see the new vertex, the new
// faces' planes, the best-face search -- and repeat the horizon walk, which is
// then a walk over links and bits (every lane keeps the same state and stores
// the same values).
//
// The walk makes its new faces' links at once, in the reference's slots and
// order, and their planes all together after it: nothing reads them earlier,
// except a walk that comes back to a slot that was freed and used again in the
// same pass, which computes that face's plane there.  A face the reference
// would have refused (degenerate or not convex) ends the pass as an invalid
// hull either way, and what the walk did after it is never read.
//
// A store of fewer faces or vertices than the reference's limits gives up
// (full) where the reference would go on; the pair then starts again in a
// store of the full size.
#pragma once
#include "shape64.h"

namespace fclx {
namespace shp {

// Links of a face in two words, read at once: its neighbours f (7 bits each)
// with the neighbours' edges e (2 bits each) and the walk's marks; its
// vertices c (7 bits each).
struct alignas(8) Links {
  uint32_t f, c;
};
enum : uint32_t {
  kSeen = 1u << 27,   // the face sees the pass's new vertex
  kBeen = 1u << 28,   // the walk has been to it
  kFresh = 1u << 29,  // made in this pass: its plane is not computed yet
  kMarks = kSeen | kBeen | kFresh
};
__device__ __forceinline__ int link_c(uint32_t c, int i) { return (c >> (7 * i)) & 127; }
__device__ __forceinline__ int link_f(uint32_t f, int i) { return (f >> (7 * i)) & 127; }
__device__ __forceinline__ int link_e(uint32_t f, int i) { return (f >> (21 + 2 * i)) & 3; }
__device__ __forceinline__ uint32_t link_set(uint32_t k, int i, int f, int e) {
  const uint32_t m = (127u << (7 * i)) | (3u << (21 + 2 * i));
  return (k & ~m) | (static_cast<uint32_t>(f) << (7 * i)) |
         (static_cast<uint32_t>(e) << (21 + 2 * i));
}

// v of the lane that a butterfly step over groups of 2 * kStep lanes pairs this
// one with (within a row of 16 by DPP, which takes no LDS).
template <int kStep>
__device__ __forceinline__ int paired(int v) {
  if constexpr (kStep == 1) return __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false);
  if constexpr (kStep == 2) return __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false);
  if constexpr (kStep == 4) return __builtin_amdgcn_update_dpp(v, v, 0x141, 0xF, 0xF, false);
  if constexpr (kStep == 8) return __builtin_amdgcn_update_dpp(v, v, 0x140, 0xF, 0xF, false);
  if constexpr (kStep >= 16) return __shfl_xor(v, kStep);
}
template <int kStep>
__device__ __forceinline__ double paired(double v) {
  union {
    double d;
    int i[2];
  } u{v};
  u.i[0] = paired<kStep>(u.i[0]);
  u.i[1] = paired<kStep>(u.i[1]);
  return u.d;
}

template <int kF, int kV>
struct EpaStore {
  static constexpr int kFaces = kF, kVerts = kV;
  D3 n[kF];
  double d[kF];
  D3 w[kV];    // support points (GJK's simplex first)
  D3 dir[kV];  // their search directions
  Links k[kF];
  int16_t stamp[kF];  // append order on the hull (-1: not on it)
  int16_t xs[kF];     // horizon walk stack: face | edge << 7 | stage << 9
  uint8_t freed[kF];  // stack of freed face slots
  uint8_t made[kF];   // the pass's new faces
  MDiff m;            // the pair's Minkowski difference
  int32_t pad[4];     // groups start on different banks
};

template <int G>
struct EpaGroup {
  int lane;   // in the group
  int first;  // the group's first lane in its wavefront
  int nfreed, top_free, hi, next_stamp, nextsv, status, best, it, fb_vertex;
  bool fallback;
  bool full;  // the store is used up before the reference's limits are

  template <int kStep>
  __device__ __forceinline__ static void larger_dot(double& dt, int& at) {
    const double od = paired<kStep>(dt);
    const int oa = paired<kStep>(at);
    if (oa >= 0 && (at < 0 || od > dt || (od == dt && oa < at))) {
      dt = od;
      at = oa;
    }
  }
  // the first vertex of largest d . v, the vertices shared out over the lanes
  __device__ __forceinline__ D3 support(const Shape& s, const D3& d) const {
    if (s.type != kConvex) return shp::support(s, d);
    double maxdot = -1.7976931348623157e308;
    int at = -1;
    for (int i = lane; i < s.nv; i += G) {
      const double dt = dot(d, mk(s.verts[3 * i], s.verts[3 * i + 1], s.verts[3 * i + 2]));
      if (dt > maxdot) {
        maxdot = dt;
        at = i;
      }
    }
    if constexpr (G > 1) larger_dot<1>(maxdot, at);
    if constexpr (G > 2) larger_dot<2>(maxdot, at);
    if constexpr (G > 4) larger_dot<4>(maxdot, at);
    if constexpr (G > 8) larger_dot<8>(maxdot, at);
    if constexpr (G > 16) larger_dot<16>(maxdot, at);
    if constexpr (G > 32) larger_dot<32>(maxdot, at);
    if (at < 0) return mk(0, 0, 0);
    return mk(s.verts[3 * at], s.verts[3 * at + 1], s.verts[3 * at + 2]);
  }
  __device__ __forceinline__ D3 msupport(const MDiff& m, const D3& d) const {
    return sub(support(m.s0, d), add(rotT(m.r, support(m.s1, rot(m.r, neg(d)))), m.t));
  }

  // the stock: freed slots (the top one also in a register), then unused ones
  template <typename S>
  __device__ __forceinline__ void drop(S& M, int f) {  // off the hull, into the stock
    M.stamp[f] = -1;
    M.freed[nfreed++] = static_cast<uint8_t>(f);
    top_free = f;
  }
  template <typename S>
  __device__ __forceinline__ void bind(S& M, int fa, int ea, int fb, int eb) {
    M.k[fa].f = link_set(M.k[fa].f, ea, fb, eb);
    M.k[fb].f = link_set(M.k[fb].f, eb, fa, ea);
  }

  // epa-inl.h:145-189 newFace, in two parts: the slot (-1: none left), its
  // links to be stored ...
  template <typename S>
  __device__ __forceinline__ int take_face(S& M, int a, int b, int c, Links& k) {
    int f;
    if (nfreed > 0) {
      f = top_free;
      --nfreed;
      top_free = M.freed[nfreed > 0 ? nfreed - 1 : 0];
    } else if (hi < S::kFaces) {
      f = hi++;
    } else {
      full = S::kFaces < kNfEpa;
      status = kEpaOutOfFaces;
      return -1;
    }
    k.f = kFresh;
    k.c = static_cast<uint32_t>(a | (b << 7) | (c << 14));
    M.stamp[f] = static_cast<int16_t>(next_stamp++);
    return f;
  }
  // ... and the plane (false: refused)
  template <typename S>
  __device__ __forceinline__ bool face_plane(S& M, int f, bool forced, double tol) const {
    const uint32_t c = M.k[f].c;
    const D3 wa = M.w[link_c(c, 0)], wb = M.w[link_c(c, 1)], wc = M.w[link_c(c, 2)];
    const D3 n = cross(sub(wb, wa), sub(wc, wa));
    const double l = nrm(n);
    if (!(l > tol)) return false;
    double d;
    if (!(edge_dist(wa, wb, n, d) || edge_dist(wb, wc, n, d) || edge_dist(wc, wa, n, d)))
      d = dot(wa, n) / l;
    M.d[f] = d;
    M.n[f] = dvd(n, l);
    return forced || d >= -tol;
  }
  // the planes of the first `count` faces in made, a lane each
  template <typename S>
  __device__ __forceinline__ bool planes(S& M, int count, double tol) const {
    bool ok = true;
    for (int i = lane; i < count; i += G) ok = face_plane(M, M.made[i], false, tol) && ok;
    const unsigned long long bad = __ballot(!ok) >> first;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // read by all lanes from here on
    return (G == 64 ? bad : bad & ((1ULL << (G & 63)) - 1ULL)) == 0;
  }

  template <int kStep>
  __device__ __forceinline__ static void nearer_face(int& root, int& at, int& stamp, double& dsq) {
    const int r = paired<kStep>(root), oa = paired<kStep>(at), os = paired<kStep>(stamp);
    const double od = paired<kStep>(dsq);
    root = r > root ? r : root;
    if (oa >= 0 && (at < 0 || od < dsq || (od == dsq && os > stamp))) {
      at = oa;
      dsq = od;
      stamp = os;
    }
  }
  // epa-inl.h:193-209 findBest: the smallest d * d, ties to the latest
  // append; a NaN root (the latest append) is never displaced
  template <typename S>
  __device__ __forceinline__ int find_best(const S& M) const {
    int root = -1;  // stamp << 8 | face
    int at = -1, at_stamp = -1;
    double at_dsq = 0;
    for (int f = lane; f < hi; f += G) {
      const int s = M.stamp[f];
      if (s < 0) continue;
      const double d = M.d[f], v = d * d;
      const int r = (s << 8) | f;
      root = r > root ? r : root;
      if (v == v && (at < 0 || v < at_dsq || (v == at_dsq && s > at_stamp))) {
        at = f;
        at_dsq = v;
        at_stamp = s;
      }
    }
    if constexpr (G > 1) nearer_face<1>(root, at, at_stamp, at_dsq);
    if constexpr (G > 2) nearer_face<2>(root, at, at_stamp, at_dsq);
    if constexpr (G > 4) nearer_face<4>(root, at, at_stamp, at_dsq);
    if constexpr (G > 8) nearer_face<8>(root, at, at_stamp, at_dsq);
    if constexpr (G > 16) nearer_face<16>(root, at, at_stamp, at_dsq);
    if constexpr (G > 32) nearer_face<32>(root, at, at_stamp, at_dsq);
    if (root < 0) return -1;
    const double rd = M.d[root & 255];
    return (rd * rd != rd * rd || at < 0) ? (root & 255) : at;
  }

  // One pass's walk (epa-inl.h:347-396 expand).
  struct Walk {
    Horizon h{-1, -1, 0};
    int made = 0;
  };

  template <typename S>
  __device__ __forceinline__ bool expand(S& M, Walk& W, int w, int f0, int e0,
                                         double tol) {
    int sp = 0, f = f0, e = e0;
    int frame = 0;  // the top frame; those below it at xs[1 .. sp - 1]
    bool result = false, call = true;
    while (true) {
      if (call) {
        result = false;
        Links F = M.k[f];
        if ((F.f & kBeen) == 0) {
          const int e1 = next3(e);
          if ((F.f & kFresh) != 0) {  // a slot used again in this pass
            if (!face_plane(M, f, false, tol)) return false;
            F.f &= ~kMarks;
            if (!(dot(M.n[f], M.w[w]) - M.d[f] < -tol)) F.f |= kSeen;
            M.k[f].f = F.f;
          }
          if ((F.f & kSeen) == 0) {
            if (W.made >= S::kFaces) {
              if (!planes(M, W.made, tol)) return false;
              W.made = 0;
            }
            Links k;
            const int nf = take_face(M, link_c(F.c, e1), link_c(F.c, e), w, k);
            if (nf >= 0) {
              M.made[W.made++] = static_cast<uint8_t>(nf);
              M.k[f].f = link_set(F.f, e, nf, 0);
              k.f = link_set(k.f, 0, f, e);
              const int cf = W.h.cf;
              if (cf >= 0) {
                M.k[cf].f = link_set(M.k[cf].f, 1, nf, 2);
                k.f = link_set(k.f, 2, cf, 1);
              } else {
                W.h.ff = nf;
              }
              M.k[nf] = k;
              W.h.cf = nf;
              ++W.h.nf;
              result = true;
            }
          } else {
            M.k[f].f = F.f | kBeen;
            // every frame marks a distinct face with this pass
            if (sp >= S::kFaces) return false;
            if (sp > 0) M.xs[sp] = static_cast<int16_t>(frame);
            ++sp;
            frame = f | (e << 7) | (1 << 9);
            f = link_f(F.f, e1);
            e = link_e(F.f, e1);
            continue;  // call the first child
          }
        }
        call = false;
      }
      // return `result` to the parent frame
      if (sp == 0) return result;
      const int pf = frame & 127, pe = (frame >> 7) & 3;
      if (frame >> 9 == 1 && result) {
        frame = pf | (pe << 7) | (2 << 9);
        const int e2 = prev3(pe);
        const uint32_t F = M.k[pf].f;
        f = link_f(F, e2);
        e = link_e(F, e2);
        call = true;
        continue;  // call the second child
      }
      // a first child that failed, or both children done
      if (result) drop(M, pf);
      --sp;
      if (sp > 0) frame = M.xs[sp];
    }
  }

  // epa-inl.h:225-281 (false: the FallBack result applies, or full)
  template <typename S>
  __device__ __forceinline__ bool start(S& M, Gjk& g, const MDiff& m, double tol) {
    nfreed = top_free = hi = next_stamp = nextsv = 0;
    status = kEpaFailed;
    fallback = true;
    full = false;
    fb_vertex = 0;
    const bool enclosed = g.rank > 1 && enclose_origin(g, m);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < g.rank) {
        M.w[i] = g.w[i];
        M.dir[i] = g.d[i];
      }
    if (enclosed) {
      status = kEpaValid;
      int c0 = 0, c1 = 1;
      if (dot(sub(g.w[0], g.w[3]), cross(sub(g.w[1], g.w[3]), sub(g.w[2], g.w[3]))) < 0) {
        c0 = 1;
        c1 = 0;
        fb_vertex = 1;  // the reference swaps the simplex's first two in place
      }
      // the tetrahedron's faces (a degenerate one ends in the FallBack)
      Links k;
      (void)take_face(M, c0, c1, 2, k);
      M.k[0] = k;
      (void)take_face(M, c1, c0, 3, k);
      M.k[1] = k;
      (void)take_face(M, 2, c1, 3, k);
      M.k[2] = k;
      (void)take_face(M, c0, 2, 3, k);
      M.k[3] = k;
      bool ok = true;
#pragma unroll 1
      for (int i = 0; i < 4; ++i) ok = face_plane(M, i, true, tol) && ok;
      if (ok) {
        best = find_best(M);
        bind(M, 0, 0, 1, 0);
        bind(M, 0, 1, 2, 0);
        bind(M, 0, 2, 3, 0);
        bind(M, 1, 1, 3, 2);
        bind(M, 1, 2, 2, 1);
        bind(M, 2, 2, 3, 1);
        status = kEpaValid;
        it = 0;
        fallback = false;
        return true;
      }
    }
    status = kEpaFallBack;
    return false;
  }

  // one pass of epa-inl.h:283-321 (false once the loop has ended, or full)
  template <typename S>
  __device__ __forceinline__ bool step(S& M, const MDiff& m, double tol) {
    if (it >= 255) return false;
    ++it;
    if (nextsv >= kNvEpa) {
      status = kEpaOutOfVertices;
      return false;
    }
    if (S::kVerts < kNvGjk + kNvEpa && kNvGjk + nextsv >= S::kVerts) {
      full = true;
      return false;
    }
    const int w = kNvGjk + nextsv++;
    const int b = best;
    const D3 bn = M.n[b];
    const double bd = M.d[b];
    const uint32_t B = M.k[b].f;
    const D3 wd = normalized(bn);
    const D3 ww = msupport(m, wd);
    M.dir[w] = wd;
    M.w[w] = ww;
    if (!(dot(bn, ww) - bd > tol)) {
      status = kEpaAccuracyReached;
      return false;
    }
    for (int f = lane; f < hi; f += G) {
      const bool sees = !(dot(M.n[f], ww) - M.d[f] < -tol);
      M.k[f].f = (M.k[f].f & ~kMarks) | (sees ? kSeen : 0u) | (f == b ? kBeen : 0u);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // read by all lanes from here on
    Walk W;
    bool valid = true;
#pragma unroll 1
    for (int j = 0; j < 3 && valid; ++j)
      valid = expand(M, W, w, link_f(B, j), link_e(B, j), tol);
    if (full) return false;
    if (!(valid && W.h.nf >= 3) || !planes(M, W.made, tol)) {
      status = kEpaInvalidHull;
      return false;
    }
    bind(M, W.h.ff, 2, W.h.cf, 1);
    drop(M, b);
    best = find_best(M);
    return true;
  }

  // epa-inl.h:323-343 and the contact (gjk_solver_indep-inl.h:141-157)
  template <typename S>
  __device__ __forceinline__ Contact finish(const S& M, const MDiff& m, const Xf& tf1) const {
    D3 normal;
    double depth;
    int rank, rc0 = fb_vertex, rc1 = 0, rc2 = 0;
    double rp[3] = {1, 0, 0};
    if (fallback) {
      normal = mk(1, 0, 0);
      depth = 0;
      rank = 1;
    } else {
      const uint32_t k = M.k[best].c;
      const D3 on = M.n[best];
      const D3 projection = mul(on, M.d[best]);
      normal = on;
      depth = M.d[best];
      rank = 3;
      rc0 = link_c(k, 0);
      rc1 = link_c(k, 1);
      rc2 = link_c(k, 2);
      const D3 a = M.w[rc0], b = M.w[rc1], c2 = M.w[rc2];
      rp[0] = nrm(cross(sub(b, projection), sub(c2, projection)));
      rp[1] = nrm(cross(sub(c2, projection), sub(a, projection)));
      rp[2] = nrm(cross(sub(a, projection), sub(b, projection)));
      const double sum = rp[0] + rp[1] + rp[2];
      rp[0] /= sum;
      rp[1] /= sum;
      rp[2] /= sum;
    }
    D3 w0 = mk(0, 0, 0);
#pragma unroll 1
    for (int i = 0; i < rank; ++i) {
      const int v = i == 0 ? rc0 : (i == 1 ? rc1 : rc2);
      const double p = i == 0 ? rp[0] : (i == 1 ? rp[1] : rp[2]);
      w0 = add(w0, mul(support(m.s0, M.dir[v]), p));
    }
    Contact c;
    c.normal = normal;
    c.pos = apply(tf1, sub(w0, mul(normal, depth * 0.5)));
    c.depth = -depth;
    return c;
  }
};

// 93 % of a random batch's pairs end within the small store; the rest start
// again in the large.  Two blocks of 256 lanes a CU, split into as many groups
// as the LDS holds stores for: 32 small ones a CU, 16 large ones.  Twice the
// lanes per group at four blocks (128 registers, 109 of them spilled) took
// 5.3 + 2.1 ms where this takes 4.6 + 1.8.
using EpaSmall = EpaStore<64, 32>;
using EpaLarge = EpaStore<kNfEpa, kNvGjk + kNvEpa>;
constexpr int kEpaBlock = 256;
constexpr int kEpaBlocksPerCu = 2;
constexpr int kEpaSmallLanes = 16, kEpaLargeLanes = 32;
static_assert(kEpaBlock / kEpaSmallLanes * sizeof(EpaSmall) <= 80 * 1024 &&
                  kEpaBlock / kEpaLargeLanes * sizeof(EpaLarge) <= 80 * 1024,
              "two blocks share a CU's 160 KB of LDS");

// A wavefront's part of a block that works off a queue of `total` pairs,
// handed out by *grab; stores: the block's, one per group.  Job: load(v, m,
// g) gives entry v's Minkowski difference and GJK's final simplex, pose() the
// frame of its contact; done(contact, passes) takes the answer, spill() an
// entry that the store is too small for.
template <int G, typename Store, typename Count, typename Job>
__device__ __forceinline__ void epa_groups(Job& job, Store* stores, long long total, Count* grab,
                                           double tol) {
  const int wl = static_cast<int>(__lane_id());
  EpaGroup<G> E;
  E.lane = wl & (G - 1);
  E.first = wl - E.lane;
  Store& M = stores[threadIdx.x / G];
  const bool leads = E.lane == 0;
  long long v = -1;
  bool active = false, over = total <= 0;  // over: the queue is used up
  while (true) {
    bool fresh = false, ended = false;
    if (!over) {
      const unsigned long long idle = __ballot(!active && leads);
      if (idle != 0) {
        const int leader = __ffsll(static_cast<long long>(idle)) - 1;
        Count b = 0;
        if (wl == leader) b = atomicAdd(grab, static_cast<Count>(__popcll(idle)));
        const long long base = static_cast<long long>(__shfl(b, leader));
        over = base + __popcll(idle) >= total;
        if (!active) {
          v = base + __popcll(idle & ((1ULL << (wl - E.lane)) - 1ULL));
          if (v < total) {
            Gjk g;
            job.load(v, M.m, g);
            active = E.start(M, g, M.m, tol);
            ended = !active;
            fresh = true;
          }
        }
      }
    }
    if (active && !fresh) {
      active = E.step(M, M.m, tol);
      ended = !active;
    }
    if (ended) {
      if (E.full) {
        if (leads) job.spill();
      } else {
        const Contact c = E.finish(M, M.m, job.pose());
        if (leads) job.done(c, E.fallback ? 0 : E.it);
      }
    }
    if (over && __ballot(active) == 0) break;
  }
}

}  // namespace shp
}  // namespace fclx
