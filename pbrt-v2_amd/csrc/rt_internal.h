// rt_internal.h -- host-side declarations shared by the C ABI and the kernel launchers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "rt_search.h"

struct rt_ctx {
  int device;
  uint32_t* d_flags;  // RT_FLAG_* recorded by the traversal kernels (rt_ctx_check)
};
struct rt_scene;

namespace rti {

// Scratch in bytes of tracing a W x H image of primary rays and one of shadow rays on `s` with the
// built-in routing, where scene_check_image accepts it.
uint64_t scene_scratch(const rt_scene* s, int W, int H);
// RT_OK when `s` can trace a W x H ray image through the batched form (a rayhierarchy or
// ray-bvh scene with its BVH, a hierarchy shape the kernels support), else the status the
// batch would return.
int scene_check_image(const rt_scene* s, int W, int H);

constexpr int kMaxLevels = 12;  // hierarchy levels of a ray image
constexpr int kUnitLevels = 4;  // levels of the blocks the unit kernels and the LDS build take
                                // (leaves per block <= 64, uint64 masks); deeper blocks are
                                // built in global memory and take the per-ray path
constexpr int kMaxSub = 85;     // 1 + 4 + 16 + 64 nodes in such a block's subtree
constexpr int kThreads = 256;   // work-group size of every traversal kernel
constexpr int kMaxBlockRays = 1024;      // blocks the unit kernels stage in LDS; larger
                                         // blocks always take the per-ray path
constexpr int64_t kMaxRaysPerBlock = 1 << 24;  // top-level blocks of at most 2^24 rays
constexpr int kClusterSize = 64;  // triangles per Morton cluster
// The unit queue and the per-ray chunk slots are claimed through kClaimQueues pairs of
// counters, 128 bytes apart after the first 64 words of a group's counter block (kCounterBytes
// in all): range q of the queue is taken first by the work-groups with blockIdx % kClaimQueues
// == q (those the dispatcher places on one XCD), so each counter is hit from one XCD until its
// range runs out.
constexpr int kClaimQueues = 8;
constexpr int kClaimBase = 64, kClaimStride = 32;
constexpr int kCounterBytes = 4 * (kClaimBase + kClaimStride * kClaimQueues);

// Ray batch in device memory (structure of arrays, row-major ray image).
struct RaysDev {
  const float *ox, *oy, *oz, *dx, *dy, *dz, *tmin, *tmax;
  const uint8_t* valid;
  int W, H;
};

// Shape of a ray hierarchy: levels, grid dims per level, node offsets, block geometry.
// Level 0 is the leaf level; the top level L-1 has one work-group per node ("block").
struct RHGeom {
  int W, H, cx, cy, L;
  int gw[kMaxLevels], gh[kMaxLevels], off[kMaxLevels];
  int nlx;     // leaves per block side = 1 << (L-1)
  int bw, bh;  // block size in rays
  int rb;      // rays per block
  int g;       // rays per leaf
  int nsub;    // nodes in a block subtree
  int ntop;    // number of blocks
  int nnodes;  // total nodes over all levels
};

// Returns 0 on success, nonzero when the shape is not supported.
int rh_geometry(int W, int H, int cx, int cy, int height, RHGeom* g);

// Whether the leaf build has at most one ray for each of a leaf's lanes.
inline bool one_ray_leaves(const RHGeom& g) { return g.g <= 64 && (g.g & (g.g - 1)) == 0; }

// Blocks up to which a launch has several work-groups to each for the grazing pass: 16 blocks of a
// 64 x 64 image leave most of the device idle.
constexpr uint32_t kGrazeSmall = 64;
// Clusters from which an occlusion block's number of passing ones is counted first (which one
// work-group does).
constexpr uint32_t kHeavy = 256, kHeavyBvh = 64;  // passing clusters, of four times as many
// Whether blocks of this shape have the grazing pass.
inline bool graze_shape(const RHGeom& g) { return g.L <= kUnitLevels && g.rb <= kMaxBlockRays; }

struct HitOut {
  int32_t* id;
  float *t, *u, *v, *dpdu, *dpdv;
};

// One rayhierarchy traversal job: a resident scene, a ray image and its outputs, with the
// job's scratch (hierarchy nodes, passing-cluster lists, reduction keys) in device memory.
// A launch group holds any number of jobs of one mode and node type; the kernels find their
// job from a global block or ray index (block_base / ray_base are prefix sums).
struct RhItem {
  RHGeom g;
  RaysDev r;
  const float* v9;       // original triangle order (finalize, repair)
  const float* uv6;      // or null
  const float* v9s;      // Morton-sorted traversal copy, clusters of 64
  const uint32_t* perm;  // sorted slot -> original triangle id
  const float4* cbox;    // cluster AABBs (min, max)
  const float4* tbox;    // AABB (min, max) of every sorted triangle
  const float4* tmt;     // ray-bvh: leaf-test operands (v1, e1, e2) of every triangle, original
                         // order (null for rayhierarchy)
  // per-ray path: search tree, its frame, and its triangles' records in search order (3 float4
  // each: leaf-test operands v1, e1, e2, then as bits the original triangle index and, for
  // ray-bvh, its tleaf entry).  tleaf: ray-bvh's reference BVH leaf of every original triangle
  // (bit 31 set: not the first primitive of its leaf; ~0u: in no leaf)
  const uint4* snode;
  SearchFrame sframe;
  const float4* tmts;
  const uint32_t* tleaf;
  // grazing pass: the records of the triangles of every cluster (cluster c's from gfirst[c] to
  // gfirst[c + 1]; gfirst null: 64 each), their leaf tests' operands, index and tleaf entry (as
  // tmts), the clusters' planes, and the boxes (as cbox) of every 64 clusters
  const GrazeNormal* gnormal;
  const GrazeTri* graze;
  const float4* gtest;
  const uint32_t* gfirst;
  const GrazeCluster* gcluster;
  const float4* gbox;
  uint32_t ntri;
  uint32_t nclusters;    // clusters of 64 triangles (rayhierarchy) or 64 frontier roots
  // ray-bvh: BVH nodes (2 float4 each), frontier roots (Morton-ordered; cbox holds the boxes
  // of their clusters), BVH position -> triangle id, and per node its parent and its depth
  // below its frontier root
  uint32_t nroots;
  const float4* bvh;
  const uint32_t* roots;
  const uint32_t* prim_order;
  const uint32_t* bvh_parent;
  const uint8_t* bvh_depth;
  float4* nodes;         // 4 float4 per hierarchy node
  uint32_t* clist;       // ntop x nclusters passing clusters
  uint64_t* keys;        // closest: one (t, id) key per ray
  uint32_t* repkeys;     // primary with repair: nearest repair-region t key per ray, else null
  uint8_t* occ;          // occlusion flags
  // grazing pass: per block 0, 1 when it is looked at, kGrazeHit or kGrazeMark when any of its rays has a hit
  // (null: no block of the job is looked at), and for closest hits the ray's nearest such hit in
  // blocks with one
  uint32_t* gblock;
  uint64_t* gseed;
  HitOut out;            // closest-hit outputs
  uint32_t* flags;       // the context's RT_FLAG_* word
  uint32_t block_base, ray_base;
  int32_t repair_run;
  uint32_t chunk_base;   // first per-ray chunk slot of the job (its blocks' slots follow)
  uint32_t unit_base;    // first staging slot of the job's work units (fixed per block)
  uint32_t unit_stride;  // staging slots per block: the most units a block can make
  int32_t gsliced;       // the group's RhGroup::graze is 2
};

constexpr uint32_t kGrazeHit = 2;
constexpr uint32_t kGrazeMark = 3;  // the same, and some ray has a repair-region hit at tmin

// A launch group: `items` is the device copy of the job table; units, counters and the
// repair list are shared by the group's jobs.
struct RhGroup {
  const RhItem* items;
  // one job, every block per-ray: its table entry (host memory), which the build kernel takes as
  // an argument and writes to items; null: items is on the device already
  const RhItem* single;
  int nitems;
  int mode;  // 0 closest primary, 1 closest secondary, 2 occluded
  int node;  // 0 box_dir, 1 ia
  int big;   // some job has more than 256 rays per block or 4 levels
  int bvh;   // ray-bvh jobs (product traversal with the scene's BVH)
  // some job has a grazing pass; 2: several work-groups take a block from the start (the build then
  // clears its rays' results)
  int graze;
  int one_ray;  // every job's leaves hold a power of two of at most 64 rays (one_ray_leaves)
  uint32_t nblocks, nrays;
  uint4* units;       // {item, block, first cluster, count}, compacted from ustage
  uint4* ustage;      // the units of every block at fixed slots (job unit_base + block * stride)
  uint4* bunits;      // per block: {units made, first staging slot, queue slot within its
                      // scan tile, the tile's unit total (first block of a tile only)}
  uint2* rq;          // per-ray path: one slot per 64-ray chunk of every block, at the job's
                      // chunk_base + block * chunks per block + chunk: {item, block * chunks
                      // per block + chunk}, or item 0xffffffff for a block of the block path
  uint32_t* ctr;      // [0] units, [2] rays flagged for repair, [4] set when any block goes
                      // per-ray; [64 + 32 q] and [64 + 32 q + 1]: next unit and next per-ray
                      // chunk slot of range q (kClaimQueues ranges)
  uint32_t* heavy;    // grazing pass: queued blocks, their number in ctr[5]
  uint32_t* replist;  // global ray indices flagged for repair (primary with repair only)
  int per_unit;       // passing clusters per work unit
  int grid;           // work-groups of the persistent unit kernel; 0 = one per resident slot
  uint32_t max_units;  // upper bound of the group's work units
  uint32_t max_chunks;  // the group's per-ray chunk slots
  // blocks whose root passes at least this many clusters are traced ray by ray; 0 sends every
  // block with a traced ray that way without the cluster scan (job cluster lists unused)
  uint32_t ray_clusters;
  int ray_grid;  // work-groups (one wavefront each) of the per-ray kernel; 0 = resident slots
  int walk;      // per-ray walk rounds, RT_PARAM_WALK_* (0: built-in)
};
constexpr int kDefaultWalk = 3;  // what the built-in walk reads as, the v that it once was

// Search tree of the per-ray path (see rt_search_bvh.cpp): a 4-wide tree over the triangles in
// their own search order.  A node is one 64-byte line, 4 uint4:
//   [0..2]  per axis x, y, z: the children's lower planes, then their upper planes, 4 FP16 each,
//           in units of SearchFrame::unit above the node's grid cell, rounded outward
//   [3].x   grid cell of the node, 8 bits per axis from bit 0 (cell c starts at base + c * unit);
//           bits 24..31: the number of interior children ni (they come first)
//   [3].y   index of the first interior child; child i < ni is node [3].y + i
//   [3].z   kSearchLeafBit + position of the first leaf's triangle - ni, so that child i >= ni
//           is the leaf reference [3].z + i (one triangle per leaf)
//   [3].w   the number of children n (1..4): a walk enters children below n only
// A depth-first walk that keeps the unvisited children of every node on its path holds at most
// kSearchStack of them, whatever the ray: the builder counts n - 1 for a node, and the count, not
// the planes of the absent children, keeps a ray out of those (a direction or origin that is not
// finite, or an origin so far out that its slack exceeds the planes' range, passes every plane
// test).
constexpr uint32_t kSearchLeafBit = 0x80000000u;
constexpr int kSearchDepth = 26;  // interior levels of the binary tree it is collapsed from
// Entries of the walk's stack in LDS; the tree's builder keeps narrower nodes where a deeper
// stack would be needed.  The most that leaves the closest-hit kernel's work-groups (10,240 bytes
// of LDS each, handed out in 1,280-byte pieces) at 16 per CU, which its registers allow too.
// With 26 entries the nodes were a fifth more on a cluster scene (1 M segments 673 us, 626 with
// 30).
constexpr int kSearchStack = 32;
constexpr uint32_t kSearchPad = 4;  // records of zeros after the triangles'
// Builds the search tree of `ntri` triangles (v9 in the caller's order): the nodes (4 uint4
// each), the search order (position -> triangle index) and the frame of the node planes.
void build_search_bvh(const float* v9, uint32_t ntri, std::vector<uint4>& nodes,
                      std::vector<uint32_t>& order, SearchFrame& frame);

// Allocation-free trace: a static device array of kNoAllocScratch bytes per device (defined in
// rt_kernels.hip).  noalloc_setup looks up its address on `device`, which must be current
// (once per device; 0 on success); noalloc_scratch returns it (null before setup).
constexpr size_t kNoAllocScratch = (size_t)64 << 20;
constexpr int kMaxDevices = 64;
int noalloc_setup(int device);
void* noalloc_scratch(int device);
// Records of the grazing pass for the triangles order[0 .. n) of v9 (original triangle order;
// tleaf: RhItem::tleaf or null), and of the clusters that they make up: from first[c] to
// first[c + 1], or 64 each (first null).
hipError_t launch_graze_records(const float* v9, const uint32_t* order, const uint32_t* tleaf,
                                uint32_t n, const uint32_t* first, uint32_t nclusters,
                                const SearchFrame& frame, GrazeNormal* normal, GrazeTri* out,
                                float4* test, GrazeCluster* cout, hipStream_t s);
// Writes the tleaf entry of every triangle into its record in search order (RhItem::tmts).
hipError_t launch_set_tleaf(float4* tmts, const uint32_t* tleaf, uint32_t ntri, hipStream_t s);

// Launchers (all asynchronous on `s`).
hipError_t launch_fill_u8(uint8_t* p, uint8_t v, size_t n, hipStream_t s);
// rayhierarchy / ray-bvh group: fused build, grazing pass, per-ray kernel and, for primary
// rayhierarchy rays, repair.  With ray_clusters above 0: init, build, cluster (root) pass, with
// ray_clusters above 1 the units' scan and pack, persistent unit kernel, per-ray kernel and, for
// closest hits, finalize and repair.  Events that are given are recorded between.
struct RhEvents {
  hipEvent_t first = nullptr;     // before the group's first launch
  hipEvent_t trace = nullptr;     // before the first traversal kernel: grazing pass or unit kernel
  hipEvent_t ready = nullptr;     // before the unit or, without one, the per-ray kernel
  hipEvent_t ray = nullptr;       // before the per-ray kernel
  hipEvent_t ray_end = nullptr;   // after it
  hipEvent_t last = nullptr;      // after the group's last launch
};
hipError_t launch_rh_group(const RhGroup& G, hipStream_t s, const RhEvents& ev);
// Naive brute force from rays to hit records (mode 0, 1) or occlusion flags (mode 2); without
// triangles every ray misses.  naive_rule: shading frames as the naive kernels take them.
// merge: kNaiveMerge keys of scratch, used where several work-groups share out the triangles;
// scenes of under kNaiveSplit triangles need none.
constexpr uint32_t kNaiveSplit = 6144;
constexpr uint32_t kNaiveGroups = 1024;  // work-groups that a launch should have
constexpr size_t kNaiveMerge = (size_t)kNaiveGroups * 8;  // fewer have 8 rays each at most
hipError_t launch_naive_trace(const RaysDev& r, int mode, const float* v9, const float* uv6,
                              uint32_t ntri, bool naive_rule, uint64_t* merge, HitOut out,
                              uint8_t* occ, hipStream_t s);
hipError_t launch_camera_rays(int W, int H, int spp, const float origin[3], float tan_half,
                              float aspect, uint32_t seed, float* ox, float* oy, float* oz,
                              float* dx, float* dy, float* dz, float* tmin, float* tmax,
                              hipStream_t s);
hipError_t launch_bounce_rays(const RaysDev& in, const float* v9, const int32_t* id,
                              const float* t, uint32_t seed, int depth, float* ox, float* oy,
                              float* oz, float* dx, float* dy, float* dz, float* tmin,
                              float* tmax, uint8_t* valid, hipStream_t s);
// count (optional): incremented by the number of valid shadow rays written.
hipError_t launch_shadow_rays(const RaysDev& pr, const int32_t* id, const float* t, float lx,
                              float ly, float lz, float* ox, float* oy, float* oz, float* dx,
                              float* dy, float* dz, float* tmin, float* tmax, uint8_t* valid,
                              hipStream_t s, uint32_t* count = nullptr);

}  // namespace rti
