// Launch descriptors shared by the C ABI layer and the kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fclx.h"
#include "fclx_layout.h"

namespace fclx {

// bits of the context's device status word
enum : int32_t {
  kStatusStackOverflow = 1,
  kStatusPairOverflow = 2,
  kStatusQueueOverflow = 4,
  kStatusBadQuery = 8,  // a query named a missing mesh or an unsupported BV pair
  kStatusFrontOverflow = 16,  // a BVTT front outgrew its room
};

// Largest per-lane stack the traversal kernels are instantiated for; the
// host rejects meshes whose summed depths exceed it.
constexpr int kMaxStack = 256;

// Most blocks of a kernel that takes a wavefront (or part of one) per query:
// larger batches loop.  HIP refuses a launch of 2^32 threads, and by this
// size the chip's few thousand wavefront slots have long averaged out the
// queries' lengths.
constexpr int kMaxGroupBlocks = 1 << 20;
inline unsigned group_blocks(long long want) {
  return static_cast<unsigned>(want < kMaxGroupBlocks ? want : kMaxGroupBlocks);
}

struct CollideLaunch {
  const MeshDev* meshes;       // device table indexed by mesh id
  int32_t num_meshes;
  int32_t num_queries;
  const int32_t* query_meshes; // 2 per query
  const double* tf1;           // 12 per query
  const double* tf2;
  int32_t cap;                 // num_max_contacts
  int32_t* counts;             // per query
  int32_t* pairs;              // 3 per record: query, b1, b2
  long long pair_capacity;
  long long* num_pairs;        // running record count (may exceed capacity); NULL
                               // for the ordered kernel's single queries
  long long* bv_tests;         // optional, per query
  long long* leaf_tests;       // optional, per query
  int32_t* status;             // device status word (kStatus* bits)
  // enable_contact (not in the plain engine): a record per contact, with its
  // world-frame point (3), normal (3) and penetration depth
  int32_t contact;
  uint32_t carry_max;          // ordered kernel: most BV tests its list carries
  long long node_pairs_max;    // no query has more node pairs (nor BV tests)
  double* contact_pos;
  double* contact_normal;
  double* contact_depth;
  // Queries of at most this many node pairs (the product of the meshes' node
  // counts) run on a lane each, the others on lane groups: none, some of the
  // batch, or kAllLanes
  long long lanes_max;
};
constexpr long long kAllLanes = 0x7fffffffffffffffLL;
__device__ __forceinline__ long long node_pairs(const MeshDev& a, const MeshDev& b) {
  return static_cast<long long>(a.num_bvs) * b.num_bvs;
}
// lanes_max for a batch of a context whose meshes have from nodes_min to
// nodes_max nodes: limit, or what it comes to there.
inline long long lanes_within(long long limit, size_t nodes_min, size_t nodes_max) {
  if (static_cast<double>(nodes_min) * nodes_min > static_cast<double>(limit)) return 0;
  if (static_cast<double>(nodes_max) * nodes_max <= static_cast<double>(limit)) return kAllLanes;
  return limit;
}

struct DistanceLaunch {
  const MeshDev* meshes;
  int32_t num_meshes;
  int32_t num_queries;
  const int32_t* query_meshes;
  const double* tf1;
  const double* tf2;
  double* distance;            // per query
  double* points;              // optional, 6 per query (world frame)
  int32_t* ids;                // optional, 2 per query
  long long* bv_tests;
  long long* leaf_tests;
  int32_t* status;
  long long lanes_max;         // as in CollideLaunch (the plain kernel's: kAllLanes)
};

// Primitive-shape pairs (records in the fclx_shape layout of fclx.h)
struct ShapeLaunch {
  int32_t num_pairs;
  int32_t num_shapes;
  const fclx_shape* shapes;    // device, num_shapes records
  const double* vertices;      // device, convex vertex pool (3 per vertex)
  long long num_vertices;
  const int32_t* pair_shapes;  // 2 shape ids per pair
  const double* tf1;           // 12 per pair
  const double* tf2;
  int32_t cap;                 // num_max_contacts
  int32_t contact;             // enable_contact
  double tol;                  // GJK and EPA tolerance
  int32_t* counts;             // per pair
  double* contact_pos;         // 3 per slot (slot = pair * cap + i), with contact
  double* contact_normal;      // 3 per slot
  double* contact_depth;       // 1 per slot
  int32_t* passes;             // optional, 2 per pair: GJK and EPA loop passes
  int32_t* status;
};

// Mesh (BVHModel<OBBRSS>) against a primitive shape.
constexpr int kMsListDepth = 440;  // deepest mesh whose descent a list in LDS holds beside a step
constexpr size_t kMsEpaQueue = size_t(4) << 30;  // bytes of queued EPA work at most
struct MeshShapeLaunch {
  const MeshDev* meshes;        // device table indexed by mesh id
  int32_t num_meshes;
  int32_t num_queries;
  const int32_t* query_meshes;  // per query: the mesh
  const int32_t* query_shapes;  // per query: the shape record
  int32_t num_shapes;
  const fclx_shape* shapes;     // device, num_shapes records
  const double* vertices;       // device, convex vertex pool (3 per vertex)
  long long num_vertices;
  const double* tf1;            // 12 per query: the mesh's pose
  const double* tf2;            // 12 per query: the shape's pose
  int32_t cap;                  // num_max_contacts
  int32_t contact;              // enable_contact
  double tol;                   // GJK and EPA tolerance
  int32_t* counts;              // per query
  int32_t* prims;               // optional, cap per query: the contacts' triangle (b1)
  double* contact_pos;          // 3 per slot (slot = query * cap + i), with contact
  double* contact_normal;       // 3 per slot
  double* contact_depth;        // 1 per slot
  long long* stats;             // optional, 2 per query: BV tests, leaf tests
  int32_t* status;
  int32_t leaf_share;           // percent of a wavefront's lanes with a leaf that starts a
                                // leaf round (1..100; 0: 100)
  int32_t list_depth;           // at most kMsListDepth (lower in tests)
  size_t epa_queue;             // at most kMsEpaQueue (lower in tests)
  long long lanes_max;          // queries on meshes of at most this many nodes run on a lane
                                // each: none, some of the batch, or kAllLanes
  int32_t max_depth;            // deepest mesh of the context (levels)
};
// waves: register budget, 1..3 waves per SIMD
hipError_t launch_mesh_shape_collide(const MeshShapeLaunch& L, int waves, hipStream_t s);
size_t mesh_shape_epa_lane_bytes();
long long mesh_shape_lanes_max(int num_queries, int cap, size_t nodes_min, size_t nodes_max);

hipError_t launch_collide_plain(const CollideLaunch& L, int stack_need, hipStream_t s);
// a query per lane with FP32 culls, for the queries of L.lanes_max node pairs
// at most (with contact geometry on request)
hipError_t launch_collide_lanes(const CollideLaunch& L, int stack_need, hipStream_t s);
// lanes_max of a batch (kernels_ordered.hip)
long long collide_lanes_max(int num_queries, int cap, size_t nodes_min, size_t nodes_max);
// collide() in the reference's order by lane groups, any num_max_contacts,
// with contact geometry and statistics on request (kernels_ordered.hip)
hipError_t launch_collide_ordered(const CollideLaunch& L, int stack_need, hipStream_t s);

// collide() with BVTT front lists: one lane per sequence of queries
struct FrontLaunch {
  const MeshDev* meshes;
  int32_t num_meshes;
  int32_t num_sequences;
  const int32_t* seq_offsets;  // num_sequences + 1: sequence s = queries [off[s], off[s+1])
  const int32_t* query_meshes; // 2 per query
  const double* tf1;
  const double* tf2;
  int32_t cap;                 // num_max_contacts
  int32_t* counts;
  int32_t* pairs;              // 3 per record: query, b1, b2
  long long pair_capacity;
  long long* num_pairs;
  long long* bv_tests;
  long long* leaf_tests;
  int2* fronts;                // front_cap entries per sequence
  int2* second;                // front_cap entries per sequence (scratch)
  int32_t* front_sizes;        // per sequence
  int32_t* front_meshes;       // 2 per sequence: the mesh pair of its front
  int32_t front_cap;
  int32_t* status;
};
hipError_t launch_collide_front(const FrontLaunch& L, int stack_need, hipStream_t s);

// Broadphase pairs of overlapping world AABBs (kernels_broadphase.hip):
// aabbs 6 doubles per object (lower x y z, upper x y z); groups optional
// (pairs only across groups); pairs 2 per pair, ascending (lower, higher);
// *num_pairs = all pairs found (those beyond capacity are not stored).
hipError_t launch_broadphase(int n, const double* aabbs, const int32_t* groups, int32_t* pairs,
                             long long capacity, long long* num_pairs, hipStream_t s);

// Device refit of one mesh (kernels_refit.hip)
struct RefitLaunch {
  const double* new_verts;     // 3 per vertex
  double* verts;               // the mesh's vertex array (replaced)
  double* tri_verts;           // the mesh's per-triangle vertex records (rebuilt)
  const int32_t* tris;
  const int32_t* span;         // 2 per node
  const int32_t* prim_pos;     // per triangle: position in the build order
  int32_t* order;              // scratch, per position: the triangle
  ObbNode64* obb64;
  RssNode64* rss64;
  double* size64;
  ObbNode32* obb32;
  RssNode32* rss32;
  double* cmax;                // device scalar: largest |OBB centre|_1
  double* rcmax;               // device scalar: largest |RSS origin|_1
  int32_t num_verts;
  int32_t num_tris;
  int32_t num_bvs;
  int32_t bv_type;
};
// bottomup: level_nodes holds the node ids level by level (root level 0),
// level_offsets_host[l] .. [l+1] (host array of levels + 1) bounding each.
hipError_t launch_refit(const RefitLaunch& L, bool bottomup, const int32_t* level_nodes,
                        const int32_t* level_offsets_host, int levels, hipStream_t s);
// Sort buffers, the EPA queue and, once a batch of kEpaLanesMin pairs asked for
// contacts, the polytopes of its lanes (1.5 GB); one per context, used by one
// batch at a time (the caller serialises calls; batches on different streams
// are ordered through an event).
constexpr int kEpaLanesMin = 240000;
struct ShapeWorkspace;
ShapeWorkspace* shape_workspace_create(int device);
void shape_workspace_destroy(ShapeWorkspace* w);
void shape_workspace_set_epa_blocks_per_cu(ShapeWorkspace* w, int blocks);
void shape_workspace_set_epa_lanes_min(ShapeWorkspace* w, int pairs);
void shape_workspace_set_waves(ShapeWorkspace* w, int waves);
hipError_t shape_collide_run(ShapeWorkspace* w, const ShapeLaunch& L, hipStream_t s);
hipError_t launch_distance_plain(const DistanceLaunch& L, int stack_need, hipStream_t s);
// distance() in the reference's order, a wavefront per query
// (kernels_clearance.hip); its entries hold node indices below 2^26
bool distance_ordered_takes(size_t max_nodes);
long long distance_lanes_max(int num_queries, size_t nodes_min, size_t nodes_max);
hipError_t launch_distance_ordered(const DistanceLaunch& L, int stack_need, hipStream_t s);
// FAST engine: wavefront-wide search with the reference's visit order kept
// as path keys (engine_dist.hip); BVTTs deeper than 62 levels go to the
// plain kernel
struct DistanceTuning {
  int queries_per_wave = 4;  // 2, 4, 8
  int waves_per_simd = 2;    // 2, 3
  int width = 32;            // most bounds of one query per step
  int leaf_batch = 16;       // leaf pairs queued before their distances are taken
  int fp32_cull = 0;         // 1: FP32 lower bounds first, FP64 where both children stay
};
hipError_t launch_distance_wave(const DistanceLaunch& L, int stack_need, const DistanceTuning& tu,
                                hipStream_t s);

}  // namespace fclx
