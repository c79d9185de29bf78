// Broadphase on the device: every pair of objects whose world AABBs overlap
// (AABB::overlap, math/bv/AABB-inl.h: closed intervals on the three axes,
// so touching boxes overlap), the candidate list a BroadPhaseCollisionManager
// hands to its callback (broadphase_collision_manager.h:77-122).
//
// Up to kTilesMax objects: every pair is tested, 64 objects against 64 per
// wavefront tile, into bit masks (one word of 64 columns per row); the rows'
// counts are summed up and each row's bits are written at its place, so the
// pairs come out in order without a sort.
//
// More: sort and sweep.  The objects are sorted by their box's lower x; 16
// lanes walk the sorted list from an object's position while the next lower
// x does not exceed its upper x, and keep the pairs that also overlap in y
// and z (and, with groups, that join objects of different groups).  The pairs
// are then sorted by (lower index, higher index), so the output does not
// depend on the order in which slots were reserved.
//
// Bound: the tiles by FP64 compares (n^2 / 2 pairs of 6) and, below 5,000
// objects, by their launches; the sweep by the list walks and the sorts'
// passes.  Whole calls on boxes in a cube, against one lane per object walking
// the sorted list: 50 objects 180 -> 50 µs, 1,000 291 -> 49, 10,000 808 -> 96,
// 16,000 1042 -> 200, 50,000 1998 -> 1295, 200,000 9238 -> 4822.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <hipcub/hipcub.hpp>

#include "kernels.h"

namespace fclx {

namespace {

constexpr int kWave = 64;

__global__ void bp_zero(unsigned long long* p) { *p = 0; }

struct Box {
  double lo[3], hi[3];
};

__device__ __forceinline__ Box load_box(const double* aabbs, int i) {
  const double* a = aabbs + 6 * static_cast<size_t>(i);
  return Box{{a[0], a[1], a[2]}, {a[3], a[4], a[5]}};
}

// Closed intervals on three axes; an unordered (NaN) bound separates nothing.
__device__ __forceinline__ bool overlap(const Box& a, const Box& b) {
  return !(a.lo[0] > b.hi[0] || b.lo[0] > a.hi[0] || a.lo[1] > b.hi[1] || b.lo[1] > a.hi[1] ||
           a.lo[2] > b.hi[2] || b.lo[2] > a.hi[2]);
}

// ------------------------------------------------------------ sort and sweep
// A double's bits in ascending order (negative NaN first, NaN last).
__device__ __forceinline__ unsigned long long order_bits(double x) {
  const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(x));
  return (u >> 63) != 0 ? ~u : u | (1ULL << 63);
}
__device__ __forceinline__ bool comes_first(const Box& a, int i, const Box& b, int j) {
  const unsigned long long x = order_bits(a.lo[0]), y = order_bits(b.lo[0]);
  return x < y || (x == y && i < j);
}

__global__ void bp_keys(int n, const double* aabbs, double* keys, int32_t* idx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  keys[i] = aabbs[6 * static_cast<size_t>(i)];
  idx[i] = i;
}

__global__ void bp_gather(int n, const double* aabbs, const int32_t* groups, const int32_t* sorted,
                          Box* boxes, int32_t* sorted_groups) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  boxes[k] = load_box(aabbs, sorted[k]);
  if (groups) sorted_groups[k] = groups[sorted[k]];
}

// unused pair slots sort after every real (lower, higher) key
__global__ void bp_fill(uint64_t* p, long long n) {
  const long long k = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k < n) p[k] = ~0ULL;
}

constexpr int kSweepLanes = 16;

__global__ void __launch_bounds__(256) bp_sweep(int n, const Box* boxes, const int32_t* groups,
                                                const int32_t* sorted, int bits, uint64_t* out,
                                                long long capacity, unsigned long long* count) {
  const int lane = threadIdx.x % kWave, first = lane & ~(kSweepLanes - 1);
  const int step = static_cast<int>(gridDim.x * (blockDim.x / kSweepLanes));
  // (the last round's wavefronts may hold walks past the last object)
  long long k = (blockIdx.x * blockDim.x + threadIdx.x) / kSweepLanes;
  for (; __ballot(k < n) != 0; k += step) {
    bool live = k < n;
    const int at = live ? static_cast<int>(k) : n - 1;
    const Box a = boxes[at];
    const int i = sorted[at], gi = groups ? groups[at] : 0;
    for (int m0 = at + 1; __ballot(live) != 0; m0 += kSweepLanes) {
      const int m = m0 + (lane - first);
      bool end = m >= n, hit = false;
      if (live && !end) {
        const Box b = boxes[m];
        end = b.lo[0] > a.hi[0];  // sorted by lower x: no later box reaches i
        hit = !end && !(groups && groups[m] == gi) && overlap(a, b);
      }
      // lanes past the first end are past the walk
      const unsigned ends =
          static_cast<unsigned>(__ballot(end) >> first) & ((1u << kSweepLanes) - 1);
      if (ends != 0 && lane - first > __ffs(static_cast<int>(ends)) - 1) hit = false;
      if (ends != 0) live = false;
      const unsigned long long hm = __ballot(hit);
      if (hm == 0) continue;
      unsigned long long base = 0;
      const int leader = __ffsll(static_cast<long long>(hm)) - 1;
      if (lane == leader) base = atomicAdd(count, static_cast<unsigned long long>(__popcll(hm)));
      base = __shfl(base, leader);
      if (!hit) continue;
      const unsigned long long slot = base + __popcll(hm & ((1ULL << lane) - 1ULL));
      if (static_cast<long long>(slot) < capacity) {
        const int j = sorted[m];
        const uint64_t low = static_cast<uint64_t>(i < j ? i : j);
        out[slot] = (low << bits) | static_cast<uint64_t>(i < j ? j : i);
      }
    }
  }
}

__global__ void bp_unpack(const uint64_t* keys, int bits, long long n, int32_t* pairs) {
  const long long k = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint64_t v = keys[k];
  const bool used = v != ~0ULL;
  pairs[2 * k] = used ? static_cast<int32_t>(v >> bits) : -1;
  pairs[2 * k + 1] = used ? static_cast<int32_t>(v & ((1ULL << bits) - 1ULL)) : -1;
}

__global__ void bp_store_count(const unsigned long long* count, long long* num_pairs) {
  *num_pairs = static_cast<long long>(*count);
}

// ------------------------------------------------------------------- tiles
// The tiles' time depends on n alone, the sweep's on the overlaps in x.  At
// 16,000 objects the tiles take 168-200 µs; the sweep 207 µs where hardly any
// overlap in x and 500 µs in a cube of touching boxes.  At 32,000 it is 500
// against 225 and 824: beyond the line a sparse scene would lose.
constexpr int kTilesMax = 16384;  // 34 MB of masks

__global__ void bp_clear(int n, uint32_t* count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) count[i] = 0;
}

// The box of the largest ordered (not NaN) lower x, the last of them in the
// sweep's order; at < 0: there is none.  Found by the whole wavefront.
struct LastBox {
  double lo;
  int at;
};
__device__ __noinline__ LastBox last_ordered(int n, const double* aabbs) {
  unsigned long long bits = 0;
  LastBox r{0.0, -1};
  for (int k = static_cast<int>(__lane_id()); k < n; k += kWave) {
    const double lo = aabbs[6 * static_cast<size_t>(k)];
    const unsigned long long u = order_bits(lo);
    if (lo == lo && (r.at < 0 || u >= bits)) {
      bits = u;
      r = LastBox{lo, k};
    }
  }
  for (int d = 1; d < kWave; d <<= 1) {
    const unsigned long long u = __shfl_xor(bits, d);
    const LastBox o{__shfl_xor(r.lo, d), __shfl_xor(r.at, d)};
    if (o.at >= 0 && (r.at < 0 || u > bits || (u == bits && o.at > r.at))) {
      bits = u;
      r = o;
    }
  }
  return r;
}

// The sweep meets a box whose lower x is NaN (sorted last) only from objects
// whose walk no ordered lower x ends before: so does the tile test.  If any
// box between the two ends the walk, the last ordered one does.
__device__ __forceinline__ bool walk_reaches(const LastBox& last, const Box& a, int i,
                                             const Box& b, int j) {
  if (last.at < 0) return true;
  const bool i_first = comes_first(a, i, b, j);
  const Box& e = i_first ? a : b;  // the earlier of the two in the sweep
  const Box& l = i_first ? b : a;
  const int ei = i_first ? i : j, li = i_first ? j : i;
  Box c{};
  c.lo[0] = last.lo;
  return !(last.lo > e.hi[0] && comes_first(e, ei, c, last.at) && comes_first(c, last.at, l, li));
}

// Rows i0..i0+63 against columns 64 w..64 w + 63: a mask word per row.
__global__ void __launch_bounds__(256) bp_tiles(int n, int words, const double* __restrict__ aabbs,
                                                const int32_t* __restrict__ groups,
                                                unsigned long long* mask, uint32_t* count) {
  const int w = static_cast<int>(blockIdx.y) * 4 + static_cast<int>(threadIdx.x) / kWave;
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  const int i0 = static_cast<int>(blockIdx.x) * kWave;
  if (w >= words || w * kWave + kWave - 1 <= i0) return;  // only columns above the diagonal
  const int j = w * kWave + lane;
  const bool in = j < n;
  const Box b = load_box(aabbs, in ? j : n - 1);
  const int gj = groups ? groups[in ? j : n - 1] : 0;
  unsigned long long mine = 0;
  LastBox last{0.0, -1};
  bool have_last = false;
  const int rows = n - i0 < kWave ? n - i0 : kWave;
  for (int r = 0; r < rows; ++r) {
    const int i = i0 + r;
    const Box a = load_box(aabbs, i);
    bool hit = in && j > i && !(groups && groups[i] == gj) && overlap(a, b);
    const bool nan = hit && (a.lo[0] != a.lo[0] || b.lo[0] != b.lo[0]);
    if (__ballot(nan) != 0) {
      if (!have_last) last = last_ordered(n, aabbs);
      have_last = true;
      if (nan) hit = walk_reaches(last, a, i, b, j);
    }
    const unsigned long long m = __ballot(hit);
    if (lane == r) mine = m;
  }
  if (lane < rows) {
    mask[static_cast<size_t>(w) * n + i0 + lane] = mine;
    if (mine != 0) atomicAdd(&count[i0 + lane], static_cast<uint32_t>(__popcll(mine)));
  }
}

// base[i] = pairs of the rows before i; *num_pairs = all of them.
constexpr int kScan = 1024;
__global__ void __launch_bounds__(kScan) bp_scan(int n, const uint32_t* count, uint32_t* base,
                                                 long long* num_pairs) {
  __shared__ uint32_t sums[kScan / kWave];
  const int per = (n + kScan - 1) / kScan, lo = static_cast<int>(threadIdx.x) * per;
  uint32_t own = 0;
  for (int k = lo; k < lo + per && k < n; ++k) own += count[k];
  uint32_t incl = own;
  const int lane = static_cast<int>(threadIdx.x) % kWave, wave = static_cast<int>(threadIdx.x) / kWave;
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t o = __shfl_up(incl, d);
    if (lane >= d) incl += o;
  }
  if (lane == kWave - 1) sums[wave] = incl;
  __syncthreads();
  uint32_t run = incl - own;
  for (int k = 0; k < wave; ++k) run += sums[k];
  if (threadIdx.x == kScan - 1) *num_pairs = static_cast<long long>(run) + own;
  for (int k = lo; k < lo + per && k < n; ++k) {
    base[k] = run;
    run += count[k];
  }
}

// A lane writes its row's pairs in ascending order (eight mask words read at
// a time); the slots past the last pair get -1.
__global__ void __launch_bounds__(kWave) bp_expand(int n, int words, const unsigned long long* mask,
                                                   const uint32_t* count, const uint32_t* base,
                                                   const long long* num_pairs, int32_t* pairs,
                                                   long long capacity) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < n && count[i] != 0) {
    long long slot = base[i];
    for (int w0 = i / kWave; w0 < words; w0 += 8) {
      unsigned long long m[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        m[k] = w0 + k < words ? mask[static_cast<size_t>(w0 + k) * n + i] : 0;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        for (unsigned long long b = m[k]; b != 0; b &= b - 1, ++slot)
          if (slot < capacity) {
            pairs[2 * slot] = i;
            pairs[2 * slot + 1] = (w0 + k) * kWave + __ffsll(static_cast<long long>(b)) - 1;
          }
    }
  }
  for (long long k = *num_pairs + i; k < capacity;
       k += static_cast<long long>(gridDim.x) * blockDim.x) {
    pairs[2 * k] = -1;
    pairs[2 * k + 1] = -1;
  }
}

// One block of stream-ordered memory cut into pieces.
struct Pieces {
  size_t bytes = 0;
  char* base = nullptr;
  template <typename T>
  size_t add(size_t count) {
    const size_t at = bytes;
    bytes += (count * sizeof(T) + 255) / 256 * 256;
    return at;
  }
  template <typename T>
  T* get(size_t at) const {
    return reinterpret_cast<T*>(base + at);
  }
};

hipError_t run_tiles(int n, const double* aabbs, const int32_t* groups, int32_t* pairs,
                     long long capacity, long long* num_pairs, hipStream_t s) {
  const int words = (n + kWave - 1) / kWave;
  Pieces mem;
  const size_t at_mask = mem.add<unsigned long long>(static_cast<size_t>(words) * n);
  const size_t at_count = mem.add<uint32_t>(n), at_base = mem.add<uint32_t>(n);
  hipError_t e = hipMallocAsync(reinterpret_cast<void**>(&mem.base), mem.bytes, s);
  if (e != hipSuccess) return e;
  auto* mask = mem.get<unsigned long long>(at_mask);
  auto* count = mem.get<uint32_t>(at_count);
  auto* base = mem.get<uint32_t>(at_base);
  bp_clear<<<(n + 255) / 256, 256, 0, s>>>(n, count);
  bp_tiles<<<dim3(words, (words + 3) / 4), 256, 0, s>>>(n, words, aabbs, groups, mask, count);
  bp_scan<<<1, kScan, 0, s>>>(n, count, base, num_pairs);
  if (capacity > 0)
    bp_expand<<<words, kWave, 0, s>>>(n, words, mask, count, base, num_pairs, pairs, capacity);
  e = hipGetLastError();
  (void)hipFreeAsync(mem.base, s);
  return e;
}

hipError_t run_sweep(int n, const double* aabbs, const int32_t* groups, int32_t* pairs,
                     long long capacity, long long* num_pairs, hipStream_t s) {
  const int block = 256;
  const int grid = (n + block - 1) / block;
  const size_t cap = static_cast<size_t>(capacity > 0 ? capacity : 0);
  int bits = 1;
  while ((1LL << bits) < n) ++bits;
  size_t t1 = 0, t2 = 0;
  double* none = nullptr;
  int32_t* none_i = nullptr;
  uint64_t* none_k = nullptr;
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(nullptr, t1, none, none, none_i, none_i, n, 0,
                                                    64, s);
  if (e == hipSuccess && cap > 0)
    e = hipcub::DeviceRadixSort::SortKeys(nullptr, t2, none_k, none_k, static_cast<int>(cap), 0,
                                          2 * bits, s);
  if (e != hipSuccess) return e;
  Pieces mem;
  const size_t at_keys = mem.add<double>(n), at_keys2 = mem.add<double>(n);
  const size_t at_idx = mem.add<int32_t>(n), at_idx2 = mem.add<int32_t>(n);
  const size_t at_box = mem.add<Box>(n), at_grp = mem.add<int32_t>(groups ? n : 1);
  const size_t at_pk = mem.add<uint64_t>(cap), at_pk2 = mem.add<uint64_t>(cap);
  const size_t at_count = mem.add<unsigned long long>(1);
  const size_t at_tmp = mem.add<char>(std::max<size_t>(std::max(t1, t2), 1));
  e = hipMallocAsync(reinterpret_cast<void**>(&mem.base), mem.bytes, s);
  if (e != hipSuccess) return e;
  auto* count = mem.get<unsigned long long>(at_count);
  auto* sorted = mem.get<int32_t>(at_idx2);
  auto* boxes = mem.get<Box>(at_box);
  auto* sorted_groups = groups ? mem.get<int32_t>(at_grp) : nullptr;
  auto* pk = mem.get<uint64_t>(at_pk);
  auto* pk2 = mem.get<uint64_t>(at_pk2);
  const unsigned cap_grid = static_cast<unsigned>((cap + block - 1) / block);
  bp_keys<<<grid, block, 0, s>>>(n, aabbs, mem.get<double>(at_keys), mem.get<int32_t>(at_idx));
  bp_zero<<<1, 1, 0, s>>>(count);
  if (cap > 0) bp_fill<<<cap_grid, block, 0, s>>>(pk, static_cast<long long>(cap));
  e = hipcub::DeviceRadixSort::SortPairs(mem.get<char>(at_tmp), t1, mem.get<double>(at_keys),
                                         mem.get<double>(at_keys2), mem.get<int32_t>(at_idx),
                                         sorted, n, 0, 64, s);
  if (e == hipSuccess) {
    bp_gather<<<grid, block, 0, s>>>(n, aabbs, groups, sorted, boxes, sorted_groups);
    bp_sweep<<<group_blocks((static_cast<long long>(n) * kSweepLanes + block - 1) / block), block, 0,
               s>>>(n, boxes, sorted_groups, sorted, bits, pk,
                              static_cast<long long>(cap), count);
    bp_store_count<<<1, 1, 0, s>>>(count, num_pairs);
    e = hipGetLastError();
  }
  // sort the pairs found (up to the capacity): the count is only known on
  // the device, so the whole capacity is sorted, unused slots last (a real
  // key never has all of its 2 bits set: the lower index is below the higher)
  if (e == hipSuccess && cap > 0) {
    e = hipcub::DeviceRadixSort::SortKeys(mem.get<char>(at_tmp), t2, pk, pk2,
                                          static_cast<int>(cap), 0, 2 * bits, s);
    if (e == hipSuccess) {
      bp_unpack<<<cap_grid, block, 0, s>>>(pk2, bits, static_cast<long long>(cap), pairs);
      e = hipGetLastError();
    }
  }
  (void)hipFreeAsync(mem.base, s);
  return e;
}

}  // namespace

hipError_t launch_broadphase(int n, const double* aabbs, const int32_t* groups, int32_t* pairs,
                             long long capacity, long long* num_pairs, hipStream_t s) {
  if (n <= 1) {
    bp_zero<<<1, 1, 0, s>>>(reinterpret_cast<unsigned long long*>(num_pairs));
    return hipGetLastError();
  }
  return n <= kTilesMax ? run_tiles(n, aabbs, groups, pairs, capacity, num_pairs, s)
                        : run_sweep(n, aabbs, groups, pairs, capacity, num_pairs, s);
}

}  // namespace fclx
