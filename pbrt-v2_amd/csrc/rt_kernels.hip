// rt_kernels.hip -- gfx950 kernels of the ray-space accelerators.
//
// Data layout in HBM (all FP32 unless noted):
//   triangles  v9[9*ntri] (p1, p2, p3), resident per scene; uv6[6*ntri] optional
//   rays       structure of arrays ox..dz, tmin, tmax (+ valid bytes), row-major ray image
//   hierarchy  4 float4 per node {dmin|valid, dmax, omin, omax}, level-major, row-major
//   keys       one uint64 per ray: (order-preserving t bits << 32) | triangle id (block path)
//   search     64-byte four-wide nodes of FP16 planes in a grid cell's units (per-ray path)
//   bvh        2 float4 per node {ax ay az bx}{by bz primOffset nPrimitives}
//
// Work decomposition of a rayhierarchy / ray-bvh trace (a launch group of one or more jobs):
//   build     one 256-thread work-group per top-level hierarchy node ("block") builds the
//             block's leaves and levels from its rays and clears the group's counters;
//   graze     in coherent blocks, work-groups list the triangles that a ray of the block may
//             graze, where the search tree finds no hits that only rounding gives, and test them;
//   ray path  wavefronts take 64-ray chunks of every block, walk each ray through a search tree
//             of the triangles and write its hit record or occlusion flag;
//   repair    the reference's repairRun pass for the rays that were listed for it.
// With RT_PARAM_RAY_CLUSTERS_* above 0, coherent blocks take the block path instead:
//   init      clears the per-ray keys / occlusion flags and the group counters;
//   cluster   one work-group per block bounds every cluster of 64 triangles (or of 64 ray-bvh
//             frontier roots) against the block root and queues work units of a few passing
//             clusters, or the block's chunks for the ray path;
//   unit      a persistent grid (one work-group per resident slot) takes units from the queue
//             with an atomic counter, stages the unit's block of rays and subtree in LDS and
//             traverses (phases below); per-ray results are reduced in LDS and merged with
//             global atomics;
//   finalize  turns each ray's (t, id) key into id / t / u / v (+ dpdu, dpdv).
// naive is one launch, in which a work-group has its rays' whole answer, or three where few rays
// meet many triangles and several work-groups share those out (naive_shape).
// The nearest hit is the smallest (t, id) key, so the result is deterministic (ties -> smallest
// id).
#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

#include "../../include/pbrt_amd_rt.h"
#include "rt_device.h"
#include "rt_internal.h"
#include "rt_search.h"

using namespace rtd;

namespace rti {

namespace {

constexpr uint32_t kNoKey32 = 0xffffffffu;

__device__ __forceinline__ int pow4_off(int s) { return ((1 << (2 * s)) - 1) / 3; }

// Pointers known to address global memory.  Loads and stores through them compile to global_*
// instructions; a generic pointer read from a job table compiles to flat_*, whose completion
// is also counted with the LDS operations, so LDS and memory waits serialize.
#define RT_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ RT_GLOBAL T* glb(T* p) {
  return (RT_GLOBAL T*)p;
}

// float4 element i through a generic or a global pointer (the global one is read as the
// native 4-vector, which has no address-space restriction on its copy).
typedef float rt_f4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ld4(const float4* p, size_t i) { return p[i]; }
__device__ __forceinline__ float4 ld4(RT_GLOBAL const float4* p, size_t i) {
  const rt_f4 v = ((RT_GLOBAL const rt_f4*)p)[i];
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float4 ld4(RT_GLOBAL float4* p, size_t i) {
  return ld4((RT_GLOBAL const float4*)p, i);
}
typedef uint32_t rt_u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 ldu4(RT_GLOBAL const uint4* p, size_t i) {
  const rt_u4 v = ((RT_GLOBAL const rt_u4*)p)[i];
  return make_uint4(v.x, v.y, v.z, v.w);
}

template <class P>
__device__ __forceinline__ V3 ld3(P p) { return {p[0], p[1], p[2]}; }

template <class P>
__device__ __forceinline__ Tri load_tri(P v9, uint32_t i) {
  const P p = v9 + 9 * (size_t)i;
  return make_tri(ld3(p), ld3(p + 3), ld3(p + 6));
}

// Leaf-test operands of a triangle (v1, e1 = v2 - v1, e2 = v3 - v1, precomputed in FP32 on the
// host) from 3 float4 per triangle; v2/v3 are not filled (the leaf test does not read them).
// Used where triangles are reached through an index (ray-bvh leaves): three 16-byte loads in
// place of nine scalar ones.
template <class P>
__device__ __forceinline__ Tri load_mt(P tmt, uint32_t i) {
  const float4 a = ld4(tmt, 3 * (size_t)i), b = ld4(tmt, 3 * (size_t)i + 1),
               c = ld4(tmt, 3 * (size_t)i + 2);
  Tri T;
  T.v1 = {a.x, a.y, a.z};
  T.e1 = {a.w, b.x, b.y};
  T.e2 = {b.z, b.w, c.x};
  T.v2 = T.v3 = T.v1;
  return T;
}

__device__ __forceinline__ void node_store(float4* __restrict__ nodes, size_t idx, const float* b,
                                           bool valid) {
  float4* p = nodes + 4 * idx;
  p[0] = make_float4(b[0], b[1], b[2], valid ? 1.f : 0.f);
  p[1] = make_float4(b[3], b[4], b[5], 0.f);
  p[2] = make_float4(b[6], b[7], b[8], 0.f);
  p[3] = make_float4(b[9], b[10], b[11], 0.f);
}

// Leaf-major mapping of a block-local ray slot: the rays of one leaf are consecutive slots,
// so a wavefront covers whole leaves.
__device__ __forceinline__ bool slot_xy(const RHGeom& g, int K, int J, int rl, int& x, int& y,
                                        int& leaf) {
  if (rl >= g.rb) return false;
  leaf = rl / g.g;
  int q = rl - leaf * g.g;
  int lk = leaf & (g.nlx - 1), lj = leaf >> (g.L - 1);  // nlx is 2^(L-1)
  x = K * g.bw + lk * g.cx + q % g.cx;
  y = J * g.bh + lj * g.cy + q / g.cx;
  return x < g.W && y < g.H;
}

__device__ __forceinline__ void box_combine(float* a, bool& ha, const float* b, bool hb) {
  if (!hb) return;
  if (!ha) {
    for (int k = 0; k < 12; ++k) a[k] = b[k];
    ha = true;
    return;
  }
  for (int k = 0; k < 3; ++k) a[k] = fmn(a[k], b[k]);
  for (int k = 3; k < 6; ++k) a[k] = fmx(a[k], b[k]);
  for (int k = 6; k < 9; ++k) a[k] = fmn(a[k], b[k]);
  for (int k = 9; k < 12; ++k) a[k] = fmx(a[k], b[k]);
}

// Direction part of ray i: 6DB / IA keep d.  Node "box_uv" keeps (slope, d.z, 0) with the
// slope d.y/d.x, 0 when d.x == 0 (rayhconstruct5DB.cl:23,32-33); the validity-aware build
// (rayhconstructP5DB.cl:25-29,43-47,52-57) gives a ray with d.x == 0 the slope interval
// [-1, 1] and marks it as a restart: the kernel assigns that interval, dropping what the
// leaf's earlier rays gave, and later rays widen it again.
template <bool USE_VALID, bool UV>
__device__ __forceinline__ void ray_box(V3 o, V3 d, float* v, bool& restart) {
  restart = false;
  if constexpr (UV) {
    const bool flat = d.x == 0.f;
    v[0] = v[3] = flat ? 0.f : d.y / d.x;
    if (USE_VALID && flat) {
      v[0] = -1.f;
      v[3] = 1.f;
      restart = true;
    }
    v[1] = v[4] = d.z;
    v[2] = v[5] = 0.f;
  } else {
    v[0] = v[3] = d.x;
    v[1] = v[4] = d.y;
    v[2] = v[5] = d.z;
  }
  v[6] = v[9] = o.x;
  v[7] = v[10] = o.y;
  v[8] = v[11] = o.z;
}

// Merge of the rays of one leaf in the reference's read order, a before b: the component-wise
// min/max, except that a restart in b (validity-aware 5DB) replaces a's slope interval.
__device__ __forceinline__ void leaf_merge(float* a, bool& ha, bool& ra, const float* b, bool hb,
                                           bool rb) {
  if (!hb) return;
  if (!ha) {
    for (int k = 0; k < 12; ++k) a[k] = b[k];
    ha = true;
    ra = rb;
    return;
  }
  box_combine(a, ha, b, true);
  if (rb) {
    a[0] = b[0];
    a[3] = b[3];
  }
  ra = ra || rb;
}

// Value of the lane that lane ^ m names, for a value that is the same in each group of m lanes
// (so any lane of the neighbouring group will do): DPP moves within a row of 16, a permute beyond.
template <int M>
__device__ __forceinline__ int from_group(int v) {
  if constexpr (M == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false);
  if constexpr (M == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false);
  if constexpr (M == 4) return __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false);
  if constexpr (M == 8) return __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, false);
  return __shfl_xor(v, M);
}
// Merges the boxes of neighbouring groups of M lanes, the lower group's rays first, when a leaf
// has more than M lanes.
template <int M, bool RESTART>
__device__ __forceinline__ void merge_groups(float* v, bool& have, bool& restart, int lanes,
                                             int tid) {
  if (M >= lanes) return;  // uniform
  float o[12];
  for (int k = 0; k < 12; ++k) o[k] = __int_as_float(from_group<M>(__float_as_int(v[k])));
  bool ho = from_group<M>((int)have) != 0;
  bool ro = RESTART && from_group<M>((int)restart) != 0;
  if (tid & M) {  // the neighbours' rays come first: ours are merged after them
    leaf_merge(o, ho, ro, v, have, restart);
    for (int k = 0; k < 12; ++k) v[k] = o[k];
    have = ho;
    restart = ro;
  } else {
    leaf_merge(v, have, restart, o, ho, ro);
  }
}

// Boxes of the leaves of block (K, J): `store(leaf, box, have)` is called by one lane for each.
// A leaf's rays are merged in the reference's read order (row by row, left to right).  A leaf of
// g.g rays is shared by the largest power of two of at most 64 lanes that it fills: each lane
// merges g.g / lanes consecutive rays, four loads in flight, then groups of lanes merge at
// distances 1, 2, 4, ... with the lower group first, which equals the sequential read.
// One lane a leaf, as leaves of other sizes than powers of two up to 64 had it, left a 100 x 4
// leaf's 400 rays to one lane: 400 x 300 image, 86 us (primary) and 149 us (with validity), now
// 11 and 12.  The build of 4 x 4 leaves over 1024 x 1024 rays went from 28 to 24 us with the DPP
// merges; it waits for its loads (the rays once, 33.6 MB: 7 us at the rate of a large copy).
// ONE: every lane has at most one ray (leaves of a power of two of at most 64 rays).
template <bool USE_VALID, bool UV, bool ONE, class F>
__device__ __forceinline__ void build_leaves(const RHGeom& g, const RaysDev& r, int K, int J,
                                             F store) {
  const int tid = threadIdx.x;
  const int lanes = 1 << (31 - __clz(min(g.g, 64)));  // uniform
  const int each = (g.g + lanes - 1) / lanes;
  const int nleaf = g.nlx * g.nlx, top = g.L - 1;
  const int lane = tid & (lanes - 1), group = tid / lanes, groups = kThreads / lanes;
  for (int base = 0; base < nleaf; base += groups) {
    const int li = base + group;
    const int x0 = K * g.bw + (li & (g.nlx - 1)) * g.cx, y0 = J * g.bh + (li >> top) * g.cy;
    float v[12];
    bool have = false, restart = false;
    const int q0 = lane * each, qn = li < nleaf ? min(each, g.g - q0) : 0;
    int dy = q0 / g.cx, dx = q0 - dy * g.cx;
    V3 o[4], d[4];
    bool h[4];
    auto load = [&](int n, int k) {  // the lane's ray n
      const int x = x0 + dx, y = y0 + dy;
      h[k] = n < qn && x < g.W && y < g.H;
      if (h[k]) {
        const size_t i = (size_t)y * g.W + x;
        if (USE_VALID && r.valid != nullptr) h[k] = glb(r.valid)[i] != 0;
        d[k] = {glb(r.dx)[i], glb(r.dy)[i], glb(r.dz)[i]};
        o[k] = {glb(r.ox)[i], glb(r.oy)[i], glb(r.oz)[i]};
      }
      if (++dx == g.cx) {
        dx = 0;
        ++dy;
      }
    };
    auto merge = [&](int k) {
      if (!h[k]) return;
      float b[12];
      bool rb;
      ray_box<USE_VALID, UV>(o[k], d[k], b, rb);
      leaf_merge(v, have, restart, b, true, rb);
    };
    if constexpr (ONE) {
      load(0, 0);
      merge(0);
    } else {
      for (int n = 0; n < each; n += 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) load(n + k, k);
#pragma unroll
        for (int k = 0; k < 4; ++k) merge(k);
      }
    }
    if (!have)
      for (int k = 0; k < 12; ++k) v[k] = 0.f;
    constexpr bool R = USE_VALID && UV;
    merge_groups<1, R>(v, have, restart, lanes, tid);
    merge_groups<2, R>(v, have, restart, lanes, tid);
    merge_groups<4, R>(v, have, restart, lanes, tid);
    merge_groups<8, R>(v, have, restart, lanes, tid);
    merge_groups<16, R>(v, have, restart, lanes, tid);
    merge_groups<32, R>(v, have, restart, lanes, tid);
    if (lane == 0 && li < nleaf) store(li, v, have);
  }
}

// ---------------------------------------------------------------------------------------
// Fused hierarchy build: one work-group builds the leaves and every level of one block
// (rayhconstruct6DB.cl / rayhconstructP6DB.cl / rayhconstruct(P)5DB.cl + levelConstruct6DB.cl /
// levelConstructP6DB.cl / levelConstruct(P)5DB.cl folded into one launch instead of
// 1 + (height-1) launches with host waits, rayhierarchy.cpp:375-549).
template <bool USE_VALID, bool UV, bool ONE>
__device__ void build_block(const RHGeom& g, const RaysDev& r, float4* __restrict__ nodes, int b,
                            float (*sBox)[12], int* sVal) {
  const int tid = threadIdx.x;
  const int top = g.L - 1;
  const int K = b % g.gw[top], J = b / g.gw[top];
  const int nleaf = g.nlx * g.nlx;
  const int leaf_off = g.nsub - nleaf;

  build_leaves<USE_VALID, UV, ONE>(g, r, K, J, [&](int li, const float* v, bool have) {
    for (int k = 0; k < 12; ++k) sBox[leaf_off + li][k] = v[k];
    sVal[leaf_off + li] = have ? 1 : 0;
  });
  __syncthreads();
  for (int li = tid; li < nleaf; li += kThreads) {
    int gk = K * g.nlx + (li & (g.nlx - 1)), gj = J * g.nlx + (li >> top);
    if (gk < g.gw[0] && gj < g.gh[0])
      node_store(nodes, (size_t)g.off[0] + (size_t)gj * g.gw[0] + gk, sBox[leaf_off + li],
                 sVal[leaf_off + li] != 0);
  }
  for (int l = 1; l < g.L; ++l) {
    const int s = top - l, nl = 1 << s, cnl = nl * 2;
    const int soff = pow4_off(s), coff = pow4_off(s + 1);
    for (int i = tid; i < nl * nl; i += kThreads) {
      int dk = i & (nl - 1), dj = i >> s;
      float v[12];
      bool have = false;
      for (int a = 0; a < 4; ++a) {
        int c = (2 * dj + (a >> 1)) * cnl + 2 * dk + (a & 1);
        box_combine(v, have, sBox[coff + c], sVal[coff + c] != 0);
      }
      if (!have)
        for (int k = 0; k < 12; ++k) v[k] = 0.f;
      for (int k = 0; k < 12; ++k) sBox[soff + i][k] = v[k];
      sVal[soff + i] = have ? 1 : 0;
      int gk = K * nl + dk, gj = J * nl + dj;
      if (gk < g.gw[l] && gj < g.gh[l])
        node_store(nodes, (size_t)g.off[l] + (size_t)gj * g.gw[l] + gk, v, have);
    }
    __syncthreads();
  }
}

// Job of a global block index in a launch group, for an index that is uniform over the
// wavefront: the lanes read 64 jobs' block prefixes at once and count those at or below the
// index (the prefixes increase with the job), one round trip per 64 jobs instead of a binary
// search's chain of dependent loads.
__device__ __forceinline__ int find_block_item(const RhItem* __restrict__ items, int n,
                                               uint32_t gb) {
  int k = 0;
  for (int c = 0; c < n; c += 64) {
    const int j = c + (int)__lane_id();
    const int m = __popcll(__ballot(j < n && items[j].block_base <= gb));
    k += m;
    if (m < 64) break;
  }
  return k - 1;
}
// Job of a global chunk index, likewise.
__device__ __forceinline__ int find_chunk_item(const RhItem* __restrict__ items, int n,
                                               uint32_t gc) {
  int k = 0;
  for (int c = 0; c < n; c += 64) {
    const int j = c + (int)__lane_id();
    const int m = __popcll(__ballot(j < n && items[j].chunk_base <= gc));
    k += m;
    if (m < 64) break;
  }
  return k - 1;
}
// The same per lane.
__device__ __forceinline__ uint32_t find_chunk_item_lane(const RhItem* __restrict__ items, int n,
                                                         uint32_t gc) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (items[mid].chunk_base <= gc) lo = mid;
    else hi = mid - 1;
  }
  return (uint32_t)lo;
}
// Job of a global block index, per lane.
__device__ __forceinline__ uint32_t find_block_item_lane(const RhItem* __restrict__ items, int n,
                                                         uint32_t gb) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (items[mid].block_base <= gb) lo = mid;
    else hi = mid - 1;
  }
  return (uint32_t)lo;
}
// Job of a global ray index (per lane).
__device__ __forceinline__ int find_ray_item(const RhItem* __restrict__ items, int n,
                                             uint32_t gr) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (items[mid].ray_base <= gr) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Build of a block of more than kUnitLevels levels (heights of 5 and more where the image
// allows them): its subtree does not fit the LDS of build_block, so the leaves and every level
// go straight to the node array, and each level reads its four children back from it (the
// work-group's own writes, ordered by the barrier between levels).  Children outside a level's
// grid are skipped, as build_block skips the invalid ones; the merge order is the same.
template <bool USE_VALID, bool UV, bool ONE>
__device__ void build_block_deep(const RHGeom& g, const RaysDev& r, float4* __restrict__ nodes,
                                 int b) {
  const int tid = threadIdx.x;
  const int top = g.L - 1;
  const int K = b % g.gw[top], J = b / g.gw[top];
  build_leaves<USE_VALID, UV, ONE>(g, r, K, J, [&](int li, const float* v, bool have) {
    const int gk = K * g.nlx + (li & (g.nlx - 1)), gj = J * g.nlx + (li >> top);
    if (gk < g.gw[0] && gj < g.gh[0])
      node_store(nodes, (size_t)g.off[0] + (size_t)gj * g.gw[0] + gk, v, have);
  });
  __syncthreads();
  for (int l = 1; l < g.L; ++l) {
    const int nl = g.nlx >> l;
    for (int i = tid; i < nl * nl; i += kThreads) {
      const int gk = K * nl + (i & (nl - 1)), gj = J * nl + (i >> (top - l));
      if (gk >= g.gw[l] || gj >= g.gh[l]) continue;
      float v[12];
      bool have = false;
      for (int a = 0; a < 4; ++a) {
        const int ck = 2 * gk + (a & 1), cj = 2 * gj + (a >> 1);
        if (ck >= g.gw[l - 1] || cj >= g.gh[l - 1]) continue;
        const float4* p = nodes + 4 * ((size_t)g.off[l - 1] + (size_t)cj * g.gw[l - 1] + ck);
        const float4 p0 = p[0], p1 = p[1], p2 = p[2], p3 = p[3];
        const float c[12] = {p0.x, p0.y, p0.z, p1.x, p1.y, p1.z,
                             p2.x, p2.y, p2.z, p3.x, p3.y, p3.z};
        box_combine(v, have, c, p0.w != 0.f);
      }
      if (!have)
        for (int k = 0; k < 12; ++k) v[k] = 0.f;
      node_store(nodes, (size_t)g.off[l] + (size_t)gj * g.gw[l] + gk, v, have);
    }
    __syncthreads();
  }
}

// Clears a group's counters (thread i of a grid of at least 8 threads).
__device__ __forceinline__ void clear_counters(uint32_t* __restrict__ ctr, uint32_t i) {
  if (i < 8) ctr[i] = 0u;
  if (i < kClaimQueues) {
    ctr[kClaimBase + kClaimStride * i] = 0u;      // units
    ctr[kClaimBase + kClaimStride * i + 1] = 0u;  // per-ray chunk slots
  }
}

// Clears the reduction state of every job: keys, repair keys, occlusion flags, counters.
template <int MODE>
__global__ __launch_bounds__(256) void rh_init_kernel(const RhItem* __restrict__ items, int nitems,
                                                      uint32_t nrays, uint32_t* __restrict__ ctr) {
  const uint32_t gi = blockIdx.x * kThreads + threadIdx.x;
  clear_counters(ctr, gi);
  if (gi >= nrays) return;
  const RhItem& it = items[find_ray_item(items, nitems, gi)];
  const uint32_t i = gi - it.ray_base;
  if (MODE == 2) {
    it.occ[i] = 0;
  } else {
    it.keys[i] = kMissKey;
    if (MODE == 0 && it.repkeys) it.repkeys[i] = 0xffffffffu;
  }
}

// Loads the subtree of block (K, J) into LDS: sub-level s = L-1-l, row-major within it.
template <class P>
__device__ __forceinline__ void load_subtree(const RHGeom& g, int K, int J, P nodes, Node* sN,
                                             int* sV) {
  const int top = g.L - 1;
  for (int i = threadIdx.x; i < g.nsub; i += kThreads) {
    int s = 0;
    while (pow4_off(s + 1) <= i) ++s;
    int local = i - pow4_off(s), nl = 1 << s, l = top - s;
    int gk = K * nl + local % nl, gj = J * nl + local / nl;
    // the level tables are read with constant indices (scalar loads issued together) and
    // selected per lane, not loaded per lane one after another
    int gw = 0, gh = 0, off = 0;
#pragma unroll
    for (int q = 0; q < kUnitLevels; ++q) {
      if (q == l) {
        gw = g.gw[q];
        gh = g.gh[q];
        off = g.off[q];
      }
    }
    int valid = 0;
    Node n{};
    if (gk < gw && gj < gh) {
      const P p = nodes + 4 * ((size_t)off + (size_t)gj * gw + gk);
      float4 a = ld4(p, 0), b = ld4(p, 1), c = ld4(p, 2), d = ld4(p, 3);
      n.dmin = {a.x, a.y, a.z};
      n.dmax = {b.x, b.y, b.z};
      n.omin = {c.x, c.y, c.z};
      n.omax = {d.x, d.y, d.z};
      valid = a.w != 0.f;
    }
    sN[i] = n;
    sV[i] = valid;
  }
}

// ---------------------------------------------------------------------------------------
// Hierarchy x triangle traversal (intersection6DB.cl, intersection6DB2.cl, intersectionP6DB.cl,
// intersectionIA.cl), breadth first with compaction at every level, one work unit (a block and
// a few of its passing clusters) at a time.  Triangles are stored Morton-sorted in clusters of
// 64 with AABBs.
//
// The result of a ray depends only on triangles that pass the whole cull chain (the
// reference's candidate set) AND pass the leaf test.  The traversal therefore descends with
// cheap exact-conservative bounds of the culls (never false where the cull is true) and
// evaluates the exact cull chain only for (triangle, leaf) pairs in which some ray passes the
// leaf test:
//   phase A  each thread takes one triangle of the unit's clusters through the per-triangle
//            bound against the block root; survivors queue in LDS (ballot compaction);
//   phase B  queued triangles are expanded kExpand at a time into 4 (triangle, child) items
//            each, bounded in parallel and compacted again, level by level down to the leaves
//            (depth first over rounds, so each level needs one queue);
//   phase C  (triangle, leaf) pairs are expanded into (pair, ray) leaf tests over the rays
//            staged in LDS; the pairs with a passing test are compacted and get the exact cull
//            chain; the tests of verified pairs update the ray (LDS atomic min of the (t, id)
//            key / occlusion bit).
constexpr int kCluster = 64;     // triangles per cluster
constexpr float kIncoherent = 0.25f;  // mean direction spread of an incoherent block's leaves
constexpr uint32_t kNoUnit = 0xffffffffu;  // no unit left in the queue
constexpr int kQ0Cap = 1024;     // root survivors held before expansion
constexpr int kQCap = 1024;      // survivors of one expansion round
constexpr int kExpand = 256;     // parents expanded per round (4 children each, 4 per thread)

// Cluster bound: conservative for every triangle (rayhierarchy) or BVH node box (ray-bvh, whose
// cull is intersectsNode in every mode) inside [cmin, cmax].
template <int MODE, int NODE, bool BVH = false>
__device__ __forceinline__ bool cluster_bound(const Node& n, V3 cmin, V3 cmax) {
  if (NODE == 1) return cull_ia(n, cmin, cmax);
  if (NODE == 2) return bound_5db(n, cmin, cmax);
  if (MODE == 0 && !BVH) return cluster_tri(n, cmin, cmax);
  return cluster_node6(n, cmin, cmax);
}
__device__ __forceinline__ V3 tri_bmin(const Tri& T) { return vmin(vmin(T.v1, T.v2), T.v3); }
__device__ __forceinline__ V3 tri_bmax(const Tri& T) { return vmax(vmax(T.v1, T.v2), T.v3); }
// Exact-conservative bound of the cull (IA is cheap enough to be its own bound).
template <int MODE, int NODE>
__device__ __forceinline__ bool cull_bound(const Node& n, const Tri& T) {
  if (NODE == 1) return cull_ia(n, tri_bmin(T), tri_bmax(T));
  if (NODE == 2) return bound_5db(n, tri_bmin(T), tri_bmax(T));
  if (MODE == 0) return prefilter_tri(n, T);
  return prefilter_node6(n, tri_bmin(T), tri_bmax(T));
}
// Bound of sorted triangle `slot`: intersectsTri's bound needs the vertices; the others
// depend on the triangle's AABB only, which is stored per sorted triangle.
template <int MODE, int NODE, class PF, class P4>
__device__ __forceinline__ bool cull_bound_slot(const Node& n, PF v9s, P4 tbox, uint32_t slot) {
  if (MODE == 0 && NODE == 0) return prefilter_tri(n, load_tri(v9s, slot));
  const float4 lo = ld4(tbox, 2 * (size_t)slot), hi = ld4(tbox, 2 * (size_t)slot + 1);
  const V3 bmin = {lo.x, lo.y, lo.z}, bmax = {hi.x, hi.y, hi.z};
  if (NODE == 1) return cull_ia(n, bmin, bmax);
  if (NODE == 2) return bound_5db(n, bmin, bmax);
  return prefilter_node6(n, bmin, bmax);
}
// The reference's cull: intersectsTri for 6DB primary rays, else intersectsNode of the node
// type on the triangle's bounds (the 5DB kernels use it in every mode, the repair pass's
// yetAnotherIntersection5DB.cl:78 included).
template <int MODE, int NODE>
__device__ __forceinline__ bool cull_exact(const Node& n, const Tri& T) {
  if (NODE == 1) return cull_ia(n, tri_bmin(T), tri_bmax(T));
  if (NODE == 2) return cull_5db(n, tri_bmin(T), tri_bmax(T));
  if (MODE == 0) return cull_tri(n, T);
  return cull_node6(n, tri_bmin(T), tri_bmax(T));
}

// Appends `item` for the lanes with `pass` set; one LDS atomic per wavefront.
__device__ __forceinline__ void ballot_append(uint32_t* q, int* cnt, bool pass, uint32_t item) {
  const uint64_t bal = __ballot(pass);
  const int lane = __lane_id();
  const int prefix = __popcll(bal & ((1ull << lane) - 1ull));
  int base = 0;
  if (lane == 0 && bal) base = atomicAdd(cnt, __popcll(bal));
  base = __shfl(base, 0);
  if (pass) q[base + prefix] = item;
}

// Chunk cursors of the expansion levels (kept in registers, identical in every thread).
struct Cursors {
  int c0 = 0, c1 = 0, c2 = 0, c3 = 0;
  __device__ int get(int s) const { return s == 0 ? c0 : s == 1 ? c1 : s == 2 ? c2 : c3; }
  __device__ void set(int s, int v) {
    if (s == 0) c0 = v;
    else if (s == 1) c1 = v;
    else if (s == 2) c2 = v;
    else c3 = v;
  }
};

// Phase C pair state.  Closest hits: 1 = some ray of the pair passes its leaf test, | kPairOk =
// the exact cull chain holds.  Occlusion with at most 31 rays per leaf: bit r = ray r of the
// leaf passes its leaf test, kPairOk as above; the verified bits are applied without running
// the leaf test again (it is the same deterministic test on the same operands).
template <int MODE>
using PairState = typename std::conditional<MODE == 2, uint32_t, uint8_t>::type;
template <int MODE>
constexpr PairState<MODE> kPairOk = MODE == 2 ? (PairState<MODE>)0x80000000u : (PairState<MODE>)2;

template <int LMAX>
struct SubSize {
  static constexpr int value = ((1 << (2 * LMAX)) - 1) / 3;
};

template <int MODE, int RBMAX, int LMAX>
struct RhShared {
  Node sN[SubSize<LMAX>::value];
  int sV[SubSize<LMAX>::value];
  float4 sRo[RBMAX];  // origin, tmin
  float4 sRd[RBMAX];  // direction, tmax
  unsigned long long sKey[MODE == 2 ? 1 : RBMAX];
  // repair key per ray (primary), or occlusion bit per ray (shadow); a bitmask keeps the
  // occlusion kernel within the LDS of six work-groups per CU
  uint32_t sAux[MODE == 0 ? RBMAX : MODE == 2 ? (RBMAX + 31) / 32 : 1];
  uint8_t sRv[RBMAX];    // ray exists and is traced
  PairState<MODE> sPair[kQ0Cap];  // phase C pair state
  uint32_t sQ0[kQ0Cap];
  uint32_t sQ[LMAX > 1 ? LMAX - 1 : 1][kQCap];  // level s >= 1 survivors live in sQ[s - 1]
  int sCnt[kUnitLevels];
  int sSeg[kThreads / 64];  // phase C: flagged pairs of each wavefront's quarter of the list
  int sTraced, sOccluded;
};

// Marks ray `slot` occluded; true when it was not marked before.
template <class SH>
__device__ __forceinline__ bool mark_occluded(SH& sh, int slot) {
  const uint32_t bit = 1u << (slot & 31);
  return (atomicOr(&sh.sAux[slot >> 5], bit) & bit) == 0u;
}

// The exact cull chain from the block root to leaf `li` (reference candidate test).
template <int MODE, int NODE, int RBMAX, int LMAX>
__device__ __forceinline__ bool exact_chain(const RHGeom& g, const RhShared<MODE, RBMAX, LMAX>& sh,
                                            const Tri& T, int li) {
  const int top = g.L - 1;
  const int lx = li & (g.nlx - 1), ly = li >> top;
  for (int s = 0; s <= top; ++s) {
    const int sh_ = top - s;
    const int idx = pow4_off(s) + (ly >> sh_) * (1 << s) + (lx >> sh_);
    if (!sh.sV[idx] || !cull_exact<MODE, NODE>(sh.sN[idx], T)) return false;
  }
  return true;
}

// Leaf test of ray slot `slot` against T; returns whether it would update the ray.
template <int MODE, class SH>
__device__ __forceinline__ bool leaf_hit(const SH& sh, int slot, const Tri& T, float& t, float& b1,
                                         float& b2) {
  const float4 o4 = sh.sRo[slot], d4 = sh.sRd[slot];
  if (!mt_strict(V3{o4.x, o4.y, o4.z}, V3{d4.x, d4.y, d4.z}, T, t, b1, b2)) return false;
  if (MODE == 2) return t > o4.w && t < d4.w;  // intersectAllLeaves.cl:177-179
  const bool main = t > o4.w && t < __int_as_float(0x7f800000);  // intersectAllLeaves.cl:57-61
  return main || (MODE == 0 && repair_region(b1, b2) && t >= o4.w);
}

// Phase C over `n` (triangle slot, leaf) pairs.  Item = (pair, ray of its leaf): consecutive
// lanes take consecutive ray slots of one pair, so the LDS ray reads are conflict-free and
// the triangle load is a broadcast.
//
// Between C1 and C2 every wavefront moves the flagged pairs of its quarter of the list to the
// front of that quarter (in place, in list order), so that the exact cull chain of C2 runs
// with every lane on a flagged pair and C3 sees flagged pairs only.  Pairs without a passing
// leaf test cannot change a ray, so dropping them changes nothing.
template <int MODE, int NODE, int RBMAX, int LMAX, class PF, class PU>
__device__ __forceinline__ void leaf_rays(const RHGeom& g, PF v9s, PU perm, uint32_t* q, int n,
                                          RhShared<MODE, RBMAX, LMAX>& sh) {
  const int G = g.g;
  const int total = n * G;
  const bool pow2 = (G & (G - 1)) == 0;
  const int lg = __ffs(G) - 1;
  const bool masked = MODE == 2 && G <= 31;
  for (int e = threadIdx.x; e < n; e += kThreads) sh.sPair[e] = 0;
  __syncthreads();
  // C1: leaf tests; flag pairs with a passing test (occlusion: the passing rays).  A ray found
  // occluded has its sRv cleared, so it takes no further tests.
  for (int item = threadIdx.x; item < total; item += kThreads) {
    const int e = pow2 ? item >> lg : item / G;
    const uint32_t P = q[e];
    const int r = item - e * G;
    const int slot = (int)(P & 63u) * G + r;
    if (!sh.sRv[slot]) continue;
    float t, b1, b2;
    if (leaf_hit<MODE>(sh, slot, load_tri(v9s, P >> 6), t, b1, b2)) {
      if constexpr (MODE == 2) {
        if (masked) atomicOr(&sh.sPair[e], 1u << r);
        else sh.sPair[e] = 1;
      } else {
        sh.sPair[e] = 1;
      }
    }
  }
  __syncthreads();
  // Compaction: wavefront w owns list positions [w * S, min(n, (w + 1) * S)), S a multiple of
  // 64.  A flagged entry moves to a position at or below its own, and each 64-entry chunk is
  // read in full before it is written, so no entry is overwritten before it has been read.
  static_assert(kThreads == 256, "four wavefronts of 64 per work-group");
  const int lane = __lane_id();
  const int wv = threadIdx.x >> 6;
  const int S = ((n + kThreads - 1) / kThreads) * 64;
  const int s0 = wv * S, s1 = min(n, s0 + S);
  int cw = 0;
  for (int base = s0; base < s1; base += 64) {
    const int e = base + lane;
    PairState<MODE> ps = 0;
    uint32_t P = 0;
    if (e < s1) {
      ps = sh.sPair[e];
      P = q[e];
    }
    const uint64_t bal = __ballot(ps != 0);
    if (ps != 0) {
      const int d = s0 + cw + __popcll(bal & ((1ull << lane) - 1ull));
      q[d] = P;
      sh.sPair[d] = ps;
    }
    cw += __popcll(bal);
  }
  if (lane == 0) sh.sSeg[wv] = cw;
  // C2: exact cull chain of the wavefront's flagged pairs (written by this wavefront above)
  int verified = 0;
  for (int i = lane; i < cw; i += 64) {
    const int e = s0 + i;
    const PairState<MODE> ps = sh.sPair[e];
    const uint32_t P = q[e];
    const bool ok = exact_chain<MODE, NODE, RBMAX, LMAX>(g, sh, load_tri(v9s, P >> 6), (int)(P & 63u));
    sh.sPair[e] = ok ? (PairState<MODE>)(ps | kPairOk<MODE>) : (PairState<MODE>)0;
    verified |= ok;
  }
  if (!__syncthreads_or(verified)) return;
  // C3: apply the leaf tests of verified pairs.  Flagged pair j (over the four quarters in
  // order) sits at position w * S + (j - p[w]), p the prefix sums of the quarters' counts.
  const int p1 = sh.sSeg[0], p2 = p1 + sh.sSeg[1], p3 = p2 + sh.sSeg[2], nf = p3 + sh.sSeg[3];
  const int ftotal = nf * G;
  for (int item = threadIdx.x; item < ftotal; item += kThreads) {
    const int j = pow2 ? item >> lg : item / G;
    const int r = item - j * G;
    const int w = (j >= p1) + (j >= p2) + (j >= p3);
    const int e = w * S + j - (w == 0 ? 0 : w == 1 ? p1 : w == 2 ? p2 : p3);
    const PairState<MODE> ps = sh.sPair[e];
    if (!(ps & kPairOk<MODE>)) continue;
    const uint32_t P = q[e];
    const uint32_t slot_t = P >> 6;
    const int slot = (int)(P & 63u) * G + r;
    if (masked) {  // occlusion: the rays that passed in C1
      if (!((ps >> r) & 1u)) continue;
      if (mark_occluded(sh, slot)) atomicAdd(&sh.sOccluded, 1);
      sh.sRv[slot] = 0;
      continue;
    }
    if (!sh.sRv[slot]) continue;
    float t, b1, b2;
    if (!leaf_hit<MODE>(sh, slot, load_tri(v9s, slot_t), t, b1, b2)) continue;
    const float tmin = sh.sRo[slot].w;
    if (MODE == 2) {
      if (mark_occluded(sh, slot)) atomicAdd(&sh.sOccluded, 1);
      sh.sRv[slot] = 0;
    } else {
      if (t > tmin && t < __int_as_float(0x7f800000))
        atomicMin(&sh.sKey[slot], (unsigned long long)hit_key(t, (int32_t)perm[slot_t]));
      if constexpr (MODE == 0) {
        if (repair_region(b1, b2) && t >= tmin) atomicMin(&sh.sAux[slot], fkey(t));
      }
    }
  }
  __syncthreads();
}

// Phases B and C for the triangles queued in sQ0; empties the queue.
template <int MODE, int NODE, int RBMAX, int LMAX, class PF, class P4, class PU>
__device__ __forceinline__ void expand_queue(const RHGeom& g, PF v9s, P4 tbox, PU perm,
                                             RhShared<MODE, RBMAX, LMAX>& sh) {
  const int tid = threadIdx.x;
  const int top = g.L - 1;
  if (top == 0) {
    leaf_rays<MODE, NODE, RBMAX, LMAX>(g, v9s, perm, sh.sQ0, sh.sCnt[0], sh);
  } else {
    Cursors cur;
    int s = 0;
    while (true) {
      const int cnt = sh.sCnt[s];
      if (s == top) {
        leaf_rays<MODE, NODE, RBMAX, LMAX>(g, v9s, perm, sh.sQ[s - 1], cnt, sh);
        --s;
        continue;
      }
      const int c = cur.get(s);
      if (c >= cnt) {
        cur.set(s, 0);
        if (s == 0) break;
        --s;
        continue;
      }
      cur.set(s, c + kExpand);
      const int np = min(kExpand, cnt - c);
      const uint32_t* src = s == 0 ? sh.sQ0 : sh.sQ[s - 1];
      __syncthreads();
      if (tid == 0) sh.sCnt[s + 1] = 0;
      __syncthreads();
      // 4 children per parent, every thread takes children until all np * 4 are bounded (a
      // uniform trip count: the append is a wavefront ballot)
      for (int cb = 0; cb < np * 4; cb += kThreads) {
        const int ct = cb + tid;
        bool ok = false;
        uint32_t item = 0;
        if (ct < np * 4) {
          const uint32_t P = src[c + (ct >> 2)];
          const uint32_t slot_t = P >> 6;
          const int pl = (int)(P & 63u), a = ct & 3;
          const int pnl = 1 << s;
          const int dk = pl & (pnl - 1), dj = pl >> s;
          const int ch = (2 * dj + (a >> 1)) * (2 * pnl) + 2 * dk + (a & 1);
          const int ni = pow4_off(s + 1) + ch;
          item = (slot_t << 6) | (uint32_t)ch;
          if (sh.sV[ni]) ok = cull_bound_slot<MODE, NODE>(sh.sN[ni], v9s, tbox, slot_t);
        }
        ballot_append(sh.sQ[s], &sh.sCnt[s + 1], ok, item);
      }
      __syncthreads();
      ++s;
    }
  }
  if (tid == 0) sh.sCnt[0] = 0;
  __syncthreads();
}

// Cluster pass: one work-group per block (of any job of the group) tests every cluster (of
// triangles, or of ray-bvh frontier roots) against the block root (cluster bound), stores the
// passing cluster ids in the job's clist[block * nclusters + ...] and appends work units
// {job, block, first, count} of at most `per_unit` passing clusters.
//
// A block whose root passes at least `ray_clusters` clusters of a scene of at least four times
// as many, or whose leaves' ray directions spread by more than kIncoherent on average, is an
// incoherent ray group: its candidate set
// holds most (leaf, triangle) pairs, so it is queued for the per-ray path instead, as 64-ray
// chunks {job, block * chunks per block + chunk} in the block's fixed slots of the queue (no
// shared counter: thousands of blocks appending through one atomic serialise on it); the
// slots of every other block are marked empty.  ray_clusters == 0 queues every block with a
// traced ray that way without scanning the clusters, and so does a block of more than
// kMaxBlockRays rays or kUnitLevels levels (the unit kernels stage at most that much; the
// reference's own scenes use such blocks, e.g. 100x4 leaves at height 3 or 4).
template <int MODE, int NODE, bool BVH>
__global__ __launch_bounds__(256) void rh_cluster_kernel(const RhItem* __restrict__ items,
                                                         int nitems, uint4* __restrict__ ustage,
                                                         uint4* __restrict__ bunits,
                                                         uint2* __restrict__ rq,
                                                         uint32_t* __restrict__ ctr,
                                                         int per_unit, uint32_t ray_clusters) {
  __shared__ int sCnt;
  __shared__ float sSpread;
  __shared__ int sLeaves;
  const int tid = threadIdx.x;
  const int k = find_block_item(items, nitems, blockIdx.x);
  const RhItem& it = items[k];
  const RHGeom& g = it.g;
  const int top = g.L - 1;
  const int b = (int)(blockIdx.x - it.block_base);
  const int K = b % g.gw[top], J = b / g.gw[top];
  const float4* p = it.nodes + 4 * ((size_t)g.off[top] + (size_t)J * g.gw[top] + K);
  const float4 a0 = p[0], a1 = p[1], a2 = p[2], a3 = p[3];
  // this block's chunk slots: filled for the per-ray path, marked empty otherwise
  const int nch = (g.rb + 63) / 64;
  uint2* const slots = rq + it.chunk_base + (size_t)b * (size_t)nch;
  auto queue_chunks = [&](bool per_ray) {
    for (int q = tid; q < nch; q += kThreads)
      slots[q] = make_uint2(per_ray ? (uint32_t)k : 0xffffffffu,
                            (uint32_t)b * (uint32_t)nch + (uint32_t)q);
    if (per_ray && tid == 0) ctr[4] = 1u;  // the per-ray kernel has work
    if (tid == 0) bunits[blockIdx.x] = make_uint4(0u, 0u, 0u, 0u);  // block-path blocks rewrite it
  };
  if (a0.w == 0.f) {  // no traced ray below this root (uniform)
    queue_chunks(false);
    return;
  }
  Node root;
  root.dmin = {a0.x, a0.y, a0.z};
  root.dmax = {a1.x, a1.y, a1.z};
  root.omin = {a2.x, a2.y, a2.z};
  root.omax = {a3.x, a3.y, a3.z};
  if (ray_clusters == 0 || g.rb > kMaxBlockRays || g.L > kUnitLevels) {
    // to the per-ray path without the cluster scan (no cluster list needed)
    queue_chunks(true);
    return;
  }
  if (tid == 0) {
    sCnt = 0;
    sSpread = 0.f;
    sLeaves = 0;
  }
  __syncthreads();
  // mean direction spread of the block's leaves (largest component range of each leaf's ray
  // directions): near 0 for camera rays and shadow rays toward a light from nearby points,
  // large for random segments, diffuse bounces and shadow rays from scattered points
  if (tid < g.nlx * g.nlx) {
    const int gk = K * g.nlx + tid % g.nlx, gj = J * g.nlx + tid / g.nlx;
    if (gk < g.gw[0] && gj < g.gh[0]) {
      const float4* q = it.nodes + 4 * ((size_t)g.off[0] + (size_t)gj * g.gw[0] + gk);
      const float4 lo = q[0], hi = q[1];
      if (lo.w != 0.f) {
        // box_uv leaves hold slope and d.z intervals: the d.z range is the spread
        const float sp = NODE == 2 ? hi.y - lo.y
                                   : fmaxf(fmaxf(hi.x - lo.x, hi.y - lo.y), hi.z - lo.z);
        atomicAdd(&sSpread, sp);
        atomicAdd(&sLeaves, 1);
      }
    }
  }
  const uint32_t nclusters = it.nclusters;
  const float4* __restrict__ cbox = it.cbox;
  uint32_t* out = it.clist + (size_t)b * nclusters;
  __syncthreads();
  // incoherent: at least `ray_clusters` clusters pass in a scene of at least 4 * ray_clusters
  // clusters (in smaller scenes the block path's work is bounded by the scene), or the block's
  // leaves spread their ray directions by more than kIncoherent on average (ray_clusters above
  // 2^29: never; 1: every block with a passing cluster).  The scan stops as soon as the
  // passing count decides that (a per-ray block needs no cluster list).
  const bool wide = sLeaves > 0 && sSpread > kIncoherent * (float)sLeaves;
  const bool may_heavy = ray_clusters == 1u || (uint64_t)nclusters >= 4ull * ray_clusters;
  const uint32_t enough = (ray_clusters <= (1u << 29) && wide) ? 1u
                          : may_heavy ? ray_clusters : 0xffffffffu;
  for (uint32_t cb = 0; cb < nclusters; cb += kThreads) {
    const uint32_t ci = cb + tid;
    bool ok = false;
    if (ci < nclusters) {
      const float4 lo = cbox[2 * (size_t)ci], hi = cbox[2 * (size_t)ci + 1];
      ok = cluster_bound<MODE, NODE, BVH>(root, V3{lo.x, lo.y, lo.z}, V3{hi.x, hi.y, hi.z});
    }
    ballot_append(out, &sCnt, ok, ci);
    if (enough != 0xffffffffu) {
      __syncthreads();
      if ((uint32_t)sCnt >= enough) break;  // uniform: every thread reads the same count
      __syncthreads();
    }
  }
  __syncthreads();
  const int cnt = sCnt;
  const bool heavy = (uint32_t)cnt >= ray_clusters && may_heavy;
  const bool per_ray = heavy || (ray_clusters <= (1u << 29) && cnt > 0 && wide);
  queue_chunks(per_ray);
  if (per_ray) return;
  // the block's units go to its fixed staging slots (no shared append counter: thousands of
  // blocks appending through one atomic serialise on it); rh_unit_scan_kernel and
  // rh_unit_pack_kernel pack them
  const int nu = (cnt + per_unit - 1) / per_unit;
  const uint32_t first = it.unit_base + (uint32_t)b * it.unit_stride;
  for (int u = tid; u < nu; u += kThreads)
    ustage[first + u] = make_uint4((uint32_t)k, (uint32_t)b, (uint32_t)(u * per_unit),
                                   (uint32_t)min(per_unit, cnt - u * per_unit));
  if (tid == 0) bunits[blockIdx.x] = make_uint4((uint32_t)nu, first, 0u, 0u);
}

// Packs the staged units of every block of a group into one queue in block order.
// - The scan takes tiles of 1,024 consecutive blocks, one work-group per tile and one block
//   per thread (coalesced). It scans within each wavefront by shuffles and across the 16
//   wavefronts through LDS, leaving each block's exclusive prefix within its tile in .z and
//   the tile's total in .w of the tile's first block.
// - The pack copies each block's units to their queue slots, one wavefront per block (four to
//   a work-group), so the copies of all blocks are in flight at once. Each wavefront first
//   adds up the totals of the tiles before its block's tile, one tile per lane. The wavefront
//   of the last block sets the queue's length, ctr[0].
// A single work-group walking the tiles in turn took ~37 us for the 58,000 blocks of a
// 64-scene batch.
constexpr int kScanThreads = 1024;
__global__ __launch_bounds__(kScanThreads) void rh_unit_scan_kernel(uint4* __restrict__ bunits,
                                                                    uint32_t nblocks) {
  __shared__ uint32_t sWave[kScanThreads / 64];
  const uint32_t tid = threadIdx.x, lane = __lane_id(), wave = tid >> 6;
  const uint32_t b = blockIdx.x * kScanThreads + tid;
  const uint32_t n = b < nblocks ? bunits[b].x : 0u;
  uint32_t incl = n;  // inclusive prefix within the wavefront
  for (uint32_t d = 1; d < 64; d <<= 1) {
    const uint32_t v = (uint32_t)__shfl_up((int)incl, d);
    if (lane >= d) incl += v;
  }
  if (lane == 63) sWave[wave] = incl;
  __syncthreads();
  uint32_t before = 0;  // units of the earlier wavefronts of the tile
  for (uint32_t w = 0; w < wave; ++w) before += sWave[w];
  if (b < nblocks) bunits[b].z = before + incl - n;
  if (tid == 0) {  // b is the tile's first block, inside the grid's range
    uint32_t total = 0;
    for (uint32_t w = 0; w < kScanThreads / 64; ++w) total += sWave[w];
    bunits[b].w = total;
  }
}
constexpr int kPackThreads = 256;
__global__ __launch_bounds__(kPackThreads) void rh_unit_pack_kernel(
    const uint4* __restrict__ bunits, uint32_t nblocks, const uint4* __restrict__ ustage,
    uint4* __restrict__ units, uint32_t* __restrict__ ctr) {
  const uint32_t b = blockIdx.x * (kPackThreads / 64u) + (threadIdx.x >> 6);
  if (b >= nblocks) return;  // uniform within the wavefront
  const uint32_t lane = __lane_id();
  const uint4 bu = bunits[b];
  uint32_t off = 0;  // units of the earlier tiles
  for (uint32_t t = lane; t < b / (uint32_t)kScanThreads; t += 64u)
    off += bunits[(size_t)t * kScanThreads].w;
  for (int d = 32; d > 0; d >>= 1) off += (uint32_t)__shfl_xor((int)off, d);
  const uint32_t to = off + bu.z;
  for (uint32_t u = lane; u < bu.x; u += 64u) units[to + u] = ustage[bu.y + u];
  if (b == nblocks - 1 && lane == 0) ctr[0] = to + bu.x;
}

// Claims the next unit of a queue of nunits split into kClaimQueues contiguous ranges with a
// counter each.  Work-group w starts in range w % kClaimQueues: the hardware deals
// work-groups to the 8 XCDs in turn, so each XCD works through its own range of blocks in its
// own L2, and one counter serves an eighth of the claims (claims of one counter serialise).
// A work-group whose range is used up moves on to the next.  Returns nunits when none is left.
// One thread of the work-group calls it and keeps the state.  word 0 selects the unit counters,
// word 1 those of the per-ray chunk slots.
// A queue that gives every work-group at most one unit is dealt by position, in the same
// eighths: no atomics, where every work-group otherwise ends with eight failing ones, on
// counters that all of them visit (~11 ns each, one after another).  Measured per-ray, 4,096
// chunks: torus 512 x 512 closest 142 -> 125 us, occlusion 148 -> 118; room task path depth 3,
// secondary 1,750 -> 1,514, occlusion 1,280 -> 1,090.  Dealing only the first units of longer
// queues by position was slower (1 M segments 680 -> 714 us): a work-group that does not start
// at once holds its unit until another one has ended.  So was reading all eight counters after
// a failed claim to go straight to a range with units left (778 us; torus occlusion units 205 ->
// 267): near the end many work-groups see the same few units, and the reads contend with the
// claims.
struct UnitClaim {
  uint32_t q, tried;
};
__device__ __forceinline__ UnitClaim claim_start() {
  return UnitClaim{blockIdx.x % (uint32_t)kClaimQueues, 0u};
}
__device__ __forceinline__ uint32_t claim_unit(uint32_t* ctr, uint32_t nunits, UnitClaim& c,
                                               int word = 0) {
  const uint32_t per = (nunits + (uint32_t)kClaimQueues - 1u) / (uint32_t)kClaimQueues;
  if (per * (uint32_t)kClaimQueues <= gridDim.x) {
    const uint32_t k = blockIdx.x / (uint32_t)kClaimQueues;
    const uint32_t u = c.tried == 0 && k < per ? c.q * per + k : nunits;
    c.tried = kClaimQueues;
    return min(u, nunits);
  }
  while (c.tried < (uint32_t)kClaimQueues) {
    const uint32_t lo = (uint32_t)((uint64_t)nunits * c.q / kClaimQueues);
    const uint32_t hi = (uint32_t)((uint64_t)nunits * (c.q + 1) / kClaimQueues);
    const uint32_t u = lo + atomicAdd(&ctr[kClaimBase + kClaimStride * c.q + word], 1u);
    if (u < hi) return u;
    c.q = (c.q + 1) % kClaimQueues;
    ++c.tried;
  }
  return nunits;
}

// Persistent unit kernel: a fixed grid takes units from the group's queue with an atomic
// counter (work stealing across every job of the group).  A unit stages its block's rays and
// subtree, takes the triangles of its clusters through the per-triangle bound (phase A),
// expands the survivors (phase B), runs the verified leaf tests (phase C) and merges the block
// results into the job's per-ray keys / occlusion flags with atomics.
template <int MODE, int NODE, int RBMAX, int LMAX>
__global__ __launch_bounds__(256) void rh_unit_kernel(const RhItem* __restrict__ items,
                                                      const uint4* __restrict__ units,
                                                      uint32_t* __restrict__ ctr) {
  __shared__ RhShared<MODE, RBMAX, LMAX> sh;
  __shared__ uint4 sUnit;  // the unit taken next; x = kNoUnit when the queue is empty
  const int tid = threadIdx.x;
  const uint32_t nunits = __builtin_amdgcn_readfirstlane(ctr[0]);
  if (nunits == 0) return;  // every block went to the per-ray path (or had no work)
  UnitClaim claim = claim_start();
  if (tid == 0) {
    const uint32_t u = claim_unit(ctr, nunits, claim);
    sUnit = u < nunits ? units[u] : make_uint4(kNoUnit, 0u, 0u, 0u);
  }
  if (tid < kUnitLevels) sh.sCnt[tid] = 0;
  if (tid == 0) {
    sh.sTraced = 0;
    sh.sOccluded = 0;
  }
  __syncthreads();
  for (;;) {
    const uint4 unit = make_uint4(__builtin_amdgcn_readfirstlane(sUnit.x),
                                  __builtin_amdgcn_readfirstlane(sUnit.y),
                                  __builtin_amdgcn_readfirstlane(sUnit.z),
                                  __builtin_amdgcn_readfirstlane(sUnit.w));
    if (unit.x == kNoUnit) break;
    const RhItem& it = items[unit.x];
    const RHGeom& g = it.g;
    const RaysDev& r = it.r;
    const auto v9s = glb(it.v9s);
    const auto perm = glb(it.perm);
    const auto tbox = glb(it.tbox);
    const uint32_t ntri = it.ntri;
    const int top = g.L - 1;
    const int b = (int)unit.y;
    const int K = b % g.gw[top], J = b / g.gw[top];
    const auto cl = glb(it.clist) + (size_t)b * it.nclusters + unit.z;
    const int ncl = (int)unit.w;
    // first cluster of this thread, loaded with the staging loads
    const uint32_t cfirst = tid / kCluster < ncl ? cl[tid / kCluster] : 0u;
    // subtree, rays, validity and occlusion flags: independent loads, issued together
    load_subtree(g, K, J, glb(it.nodes), sh.sN, sh.sV);
    for (int slot = tid; slot < RBMAX; slot += kThreads) {
      int x = 0, y = 0, leaf = 0;
      bool traced = false;
      if (slot_xy(g, K, J, slot, x, y, leaf)) {
        const size_t idx = (size_t)y * g.W + x;
        const bool valid = MODE == 0 || r.valid == nullptr || glb(r.valid)[idx] != 0;
        // a ray another unit already found occluded needs no more tests
        const bool found = MODE == 2 && glb(it.occ)[idx] != 0;
        traced = valid && !found;
        sh.sRo[slot] = make_float4(glb(r.ox)[idx], glb(r.oy)[idx], glb(r.oz)[idx],
                                   glb(r.tmin)[idx]);
        sh.sRd[slot] = make_float4(glb(r.dx)[idx], glb(r.dy)[idx], glb(r.dz)[idx],
                                   glb(r.tmax)[idx]);
      }
      sh.sRv[slot] = traced ? 1 : 0;
      if (MODE != 2) sh.sKey[slot] = kMissKey;
      if constexpr (MODE == 0) sh.sAux[slot] = kNoKey32;
      if constexpr (MODE == 2) {
        if ((slot & 31) == 0) sh.sAux[slot >> 5] = 0u;
      }
      const uint64_t bal = __ballot(traced);
      if (__lane_id() == 0 && bal) atomicAdd(&sh.sTraced, __popcll(bal));
    }
    __syncthreads();
    if (sh.sV[0] && sh.sTraced > 0) {
      const Node& root = sh.sN[0];
      bool done = false;
      for (int k0 = 0; k0 < ncl && !done; k0 += kThreads / kCluster) {
        const int k = k0 + tid / kCluster;
        const uint32_t c = k0 == 0 ? cfirst : (k < ncl ? cl[k] : 0u);
        const uint32_t slot = k < ncl ? c * kCluster + (uint32_t)(tid % kCluster) : ntri;
        bool pass = false;
        if (slot < ntri) pass = cull_bound_slot<MODE, NODE>(root, v9s, tbox, slot);
        ballot_append(sh.sQ0, &sh.sCnt[0], pass, slot << 6);
        __syncthreads();
        const int cnt0 = sh.sCnt[0];
        __syncthreads();  // every thread has read the count before the next round appends
        if (cnt0 > kQ0Cap - kThreads) {
          expand_queue<MODE, NODE, RBMAX, LMAX>(g, v9s, tbox, perm, sh);
          if (MODE == 2 && sh.sOccluded >= sh.sTraced) done = true;
        }
      }
      if (!done && sh.sCnt[0] > 0) expand_queue<MODE, NODE, RBMAX, LMAX>(g, v9s, tbox, perm, sh);
    }
    // The next unit is claimed once this one's traversal is over (a claim made earlier would
    // hold a second unit per work-group when the queue runs dry); the atomic and the
    // descriptor load overlap the merge below.
    uint4 ndesc = make_uint4(kNoUnit, 0u, 0u, 0u);
    if (tid == 0) {
      const uint32_t next = claim_unit(ctr, nunits, claim);
      if (next < nunits) ndesc = units[next];
    }
    for (int slot = tid; slot < g.rb; slot += kThreads) {
      int x, y, leaf;
      if (!slot_xy(g, K, J, slot, x, y, leaf)) continue;
      const size_t idx = (size_t)y * g.W + x;
      if (MODE == 2) {
        if ((sh.sAux[slot >> 5] >> (slot & 31)) & 1u) glb(it.occ)[idx] = 1;
      } else {
        const unsigned long long key = sh.sKey[slot];
        if (key != kMissKey) atomicMin((unsigned long long*)&it.keys[idx], key);
        if constexpr (MODE == 0) {
          if (it.repkeys) {
            const uint32_t rk = sh.sAux[slot];
            if (rk != kNoKey32) atomicMin(&it.repkeys[idx], rk);
          }
        }
      }
    }
    __syncthreads();  // LDS is rewritten by the next unit
    if (tid == 0) {
      sUnit = ndesc;
      sh.sTraced = 0;
      sh.sOccluded = 0;
    }
    if (tid < kUnitLevels) sh.sCnt[tid] = 0;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------
// ray-bvh as a launch group (intersection6DB_BVH.cl, intersection6DB_BVH2.cl,
// intersectionP6DB_BVH.cl).  The reference walks, for every block root and every frontier
// root of the CPU-built BVH, the product of the block's hierarchy and the root's BVH subtree
// in lockstep (both descend while interior; a leaf waits for the other side), culling each
// (hierarchy node, BVH node) pair with intersectsNode / the IA test, and tests the triangles
// of every (hierarchy leaf, BVH leaf) pair it reaches (only the first one for secondary rays).
// A (leaf, BVH leaf) pair is reached iff every pair on its unique lockstep path passes, so the
// same hit-first scheme as the rayhierarchy path applies: the traversal descends with the
// exact-conservative bound of the cull, runs the leaf tests, and evaluates the exact cull
// chain only for pairs in which some ray passes its leaf test.
constexpr int kBvhQCap = 3072;   // traversal stack: 256 + 224 * depth <= 3072 for depth <= 12
constexpr int kPairCap = 512;    // (BVH leaf, hierarchy leaf) pairs awaiting leaf tests
constexpr int kBvhPop = 32;      // traversal items expanded per round (8 children each)

template <int MODE, int RBMAX, int LMAX>
struct BvhShared {
  Node sN[SubSize<LMAX>::value];
  int sV[SubSize<LMAX>::value];
  float4 sRo[RBMAX];
  float4 sRd[RBMAX];
  unsigned long long sKey[MODE == 2 ? 1 : RBMAX];
  uint32_t sAux[MODE == 2 ? RBMAX : 1];  // occlusion flag (shadow)
  uint8_t sRv[RBMAX];
  uint32_t sT[kBvhQCap];   // traversal items: BVH node << 7 | subtree node index
  uint32_t sPn[kPairCap];  // pair: BVH leaf << 6 | hierarchy leaf
  // Occlusion keeps each pair's primitive range (first position, count) in LDS: its leaf
  // tests are the bulk of the work and an extra dependent load each costs more than the
  // occupancy they take.  Closest hits read the range from the leaf node, which keeps the
  // kernel within six work-groups per CU.
  uint32_t sPt[MODE == 2 ? kPairCap : 1];
  uint32_t sPc[MODE == 2 ? kPairCap : 1];
  PairState<MODE> sPair[kPairCap];  // phase C pair state
  int sSeg[kThreads / 64];  // phase C: flagged pairs of each wavefront's quarter of the list
  int sTq, sPq;
  int sTraced, sOccluded;
};

template <class P>
__device__ __forceinline__ void bvh_box(P bvh, uint32_t n, V3& bmin, V3& bmax, uint32_t& off,
                                        uint32_t& np) {
  const float4 a = ld4(bvh, 2 * (size_t)n), b = ld4(bvh, 2 * (size_t)n + 1);
  bmin = {a.x, a.y, a.z};
  bmax = {a.w, b.x, b.y};
  off = __float_as_uint(b.z);
  np = __float_as_uint(b.w);
}


template <int NODE>
__device__ __forceinline__ bool bvh_bound(const Node& n, V3 bmin, V3 bmax) {
  if (NODE == 1) return cull_ia(n, bmin, bmax);
  if (NODE == 2) return bound_5db(n, bmin, bmax);
  return prefilter_node6(n, bmin, bmax);
}
template <int NODE>
__device__ __forceinline__ bool bvh_cull(const Node& n, V3 bmin, V3 bmax) {
  if (NODE == 1) return cull_ia(n, bmin, bmax);
  if (NODE == 2) return cull_5db(n, bmin, bmax);
  return cull_node6(n, bmin, bmax);
}
// The 5DB BVH kernels skip a node with no primitives and primitive offset 0 with its subtree
// (intersection5DB_BVH.cl:18,56 and variants); the 6DB ones do not test it.
template <int NODE>
__device__ __forceinline__ bool bvh_live(uint32_t off, uint32_t np) {
  return NODE != 2 || np != 0 || off != 0;
}

// Sub-level of subtree node index i (0 root, then 4, 16, 64 nodes).
__device__ __forceinline__ int sub_level(int i) { return i == 0 ? 0 : i < 5 ? 1 : i < 21 ? 2 : 3; }

// The exact lockstep chain of the pair (BVH leaf b, hierarchy leaf li): step s visits the
// hierarchy node of level max(top - s, 0) above li and the BVH node of depth min(s, d) above b.
template <int NODE, class SH>
__device__ __forceinline__ bool bvh_chain(const RHGeom& g, const SH& sh, const RhItem& it,
                                          uint32_t b, int li) {
  const int top = g.L - 1;
  const int lx = li & (g.nlx - 1), ly = li >> top;
  const int d = (int)glb(it.bvh_depth)[b];
  uint32_t node = b;
  int dn = d;
  for (int st = max(top, d); st >= 0; --st) {
    const int bd = min(st, d);
    while (dn > bd) {
      node = glb(it.bvh_parent)[node];
      --dn;
    }
    const int ss = min(st, top);  // subtree sub-level of the hierarchy node
    const int sh_ = top - ss;
    const int idx = pow4_off(ss) + (ly >> sh_) * (1 << ss) + (lx >> sh_);
    V3 bmin, bmax;
    uint32_t off, np;
    bvh_box(glb(it.bvh), node, bmin, bmax, off, np);
    if (!bvh_live<NODE>(off, np)) return false;
    if (!sh.sV[idx] || !bvh_cull<NODE>(sh.sN[idx], bmin, bmax)) return false;
  }
  return true;
}

// First primitive position and number of primitives that pair e tests: its BVH leaf's, or
// only the first one for 6DB / IA secondary rays (intersection6DB_BVH2.cl:88; the 5DB kernel
// tests them all, intersection5DB_BVH2.cl:84).
template <int MODE, int NODE, class SH>
__device__ __forceinline__ void pair_prims(const SH& sh, const RhItem& it, int e, uint32_t& off,
                                           uint32_t& cnt) {
  if constexpr (MODE == 2) {
    off = sh.sPt[e];
    cnt = sh.sPc[e];
  } else {
    const float4 b = ld4(glb(it.bvh), 2 * (size_t)(sh.sPn[e] >> 6) + 1);
    off = __float_as_uint(b.z);
    cnt = MODE == 1 && NODE != 2 ? 1u : __float_as_uint(b.w);
  }
}

// Leaf tests of the queued pairs (test, exact chain of pairs with a passing test, apply).
template <int MODE, int NODE, int RBMAX, int LMAX>
__device__ __forceinline__ void bvh_leaf_rays(const RHGeom& g, const RhItem& it,
                                              BvhShared<MODE, RBMAX, LMAX>& sh) {
  constexpr int TM = MODE == 0 ? 1 : MODE;  // ray-bvh has no repair pass
  const int n = sh.sPq;
  const int G = g.g;
  const int total = n * G;
  const bool pow2 = (G & (G - 1)) == 0;
  const int lg = __ffs(G) - 1;
  const bool masked = MODE == 2 && G <= 31;
  for (int e = threadIdx.x; e < n; e += kThreads) sh.sPair[e] = 0;
  __syncthreads();
  for (int item = threadIdx.x; item < total; item += kThreads) {
    const int e = pow2 ? item >> lg : item / G;
    const int r = item - e * G;
    const int slot = (int)(sh.sPn[e] & 63u) * G + r;
    if (!sh.sRv[slot]) continue;  // cleared once the ray is found occluded
    uint32_t off, cnt;
    pair_prims<MODE, NODE>(sh, it, e, off, cnt);
    for (uint32_t f = 0; f < cnt; ++f) {
      float t, b1, b2;
      if (leaf_hit<TM>(sh, slot, load_mt(glb(it.tmt), glb(it.prim_order)[off + f]), t, b1,
                       b2)) {
        if constexpr (MODE == 2) {
          if (masked) atomicOr(&sh.sPair[e], 1u << r);
          else sh.sPair[e] = 1;
        } else {
          sh.sPair[e] = 1;
        }
        break;
      }
    }
  }
  __syncthreads();
  // Compaction of the flagged pairs, per wavefront and in place, as in leaf_rays.
  const int lane = __lane_id();
  const int wv = threadIdx.x >> 6;
  const int S = ((n + kThreads - 1) / kThreads) * 64;
  const int s0 = wv * S, s1 = min(n, s0 + S);
  int cw = 0;
  for (int base = s0; base < s1; base += 64) {
    const int e = base + lane;
    PairState<MODE> ps = 0;
    uint32_t pn = 0, pt = 0, pc = 0;
    if (e < s1) {
      ps = sh.sPair[e];
      pn = sh.sPn[e];
      if constexpr (MODE == 2) {
        pt = sh.sPt[e];
        pc = sh.sPc[e];
      }
    }
    const uint64_t bal = __ballot(ps != 0);
    if (ps != 0) {
      const int d = s0 + cw + __popcll(bal & ((1ull << lane) - 1ull));
      sh.sPair[d] = ps;
      sh.sPn[d] = pn;
      if constexpr (MODE == 2) {
        sh.sPt[d] = pt;
        sh.sPc[d] = pc;
      }
    }
    cw += __popcll(bal);
  }
  if (lane == 0) sh.sSeg[wv] = cw;
  int verified = 0;
  for (int i = lane; i < cw; i += 64) {
    const int e = s0 + i;
    const PairState<MODE> ps = sh.sPair[e];
    const bool ok = bvh_chain<NODE>(g, sh, it, sh.sPn[e] >> 6, (int)(sh.sPn[e] & 63u));
    sh.sPair[e] = ok ? (PairState<MODE>)(ps | kPairOk<MODE>) : (PairState<MODE>)0;
    verified |= ok;
  }
  if (__syncthreads_or(verified)) {
    const int p1 = sh.sSeg[0], p2 = p1 + sh.sSeg[1], p3 = p2 + sh.sSeg[2], nf = p3 + sh.sSeg[3];
    const int ftotal = nf * G;
    for (int item = threadIdx.x; item < ftotal; item += kThreads) {
      const int j = pow2 ? item >> lg : item / G;
      const int r = item - j * G;
      const int w = (j >= p1) + (j >= p2) + (j >= p3);
      const int e = w * S + j - (w == 0 ? 0 : w == 1 ? p1 : w == 2 ? p2 : p3);
      const PairState<MODE> ps = sh.sPair[e];
      if (!(ps & kPairOk<MODE>)) continue;
      const int slot = (int)(sh.sPn[e] & 63u) * G + r;
      if (masked) {  // occlusion: the rays that passed in C1
        if (!((ps >> r) & 1u)) continue;
        if (atomicOr(&sh.sAux[slot], 1u) == 0u) atomicAdd(&sh.sOccluded, 1);
        sh.sRv[slot] = 0;
        continue;
      }
      if (!sh.sRv[slot]) continue;
      uint32_t off, cnt;
      pair_prims<MODE, NODE>(sh, it, e, off, cnt);
      for (uint32_t f = 0; f < cnt; ++f) {
        const uint32_t tri = glb(it.prim_order)[off + f];
        float t, b1, b2;
        if (!leaf_hit<TM>(sh, slot, load_mt(glb(it.tmt), tri), t, b1, b2)) continue;
        if (MODE == 2) {
          if (atomicOr(&sh.sAux[slot], 1u) == 0u) atomicAdd(&sh.sOccluded, 1);
          sh.sRv[slot] = 0;
          break;
        }
        atomicMin(&sh.sKey[slot], (unsigned long long)hit_key(t, (int32_t)tri));
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) sh.sPq = 0;
  __syncthreads();
}

// Appends the (BVH leaf, hierarchy leaf) pair of a reached leaf x leaf pair; its primitives
// are tested together (only the first one for secondary rays, intersection6DB_BVH2.cl).
template <int MODE, class SH>
__device__ __forceinline__ void bvh_emit(SH& sh, uint32_t b, uint32_t off, uint32_t np, int li,
                                         uint32_t* flags) {
  const int e = atomicAdd(&sh.sPq, 1);
  if (e < kPairCap) {  // room for every emission of one round is kept free
    sh.sPn[e] = (b << 6) | (uint32_t)li;
    if constexpr (MODE == 2) {
      sh.sPt[e] = off;
      sh.sPc[e] = np;
    }
  } else {
    atomicOr(flags, RT_FLAG_PAIR_CAP);  // reported by rt_ctx_check
  }
}

template <int MODE, int NODE, int RBMAX, int LMAX>
__global__ __launch_bounds__(256) void bvh_unit_kernel(const RhItem* __restrict__ items,
                                                       const uint4* __restrict__ units,
                                                       uint32_t* __restrict__ ctr) {
  __shared__ BvhShared<MODE, RBMAX, LMAX> sh;
  __shared__ uint32_t sUnit;
  const int tid = threadIdx.x;
  const uint32_t nunits = __builtin_amdgcn_readfirstlane(ctr[0]);
  if (nunits == 0) return;
  UnitClaim claim = claim_start();
  for (;;) {
    if (tid == 0) sUnit = claim_unit(ctr, nunits, claim);
    __syncthreads();
    const uint32_t u = __builtin_amdgcn_readfirstlane(sUnit);
    if (u >= nunits) break;
    const uint4 unit = units[u];
    const RhItem& it = items[__builtin_amdgcn_readfirstlane(unit.x)];
    const RHGeom& g = it.g;
    const RaysDev& r = it.r;
    const int top = g.L - 1;
    const int b = (int)__builtin_amdgcn_readfirstlane(unit.y);
    const int K = b % g.gw[top], J = b / g.gw[top];
    if (tid == 0) {
      sh.sTq = 0;
      sh.sPq = 0;
      sh.sTraced = 0;
      sh.sOccluded = 0;
    }
    load_subtree(g, K, J, glb(it.nodes), sh.sN, sh.sV);
    __syncthreads();
    for (int slot = tid; slot < RBMAX; slot += kThreads) {
      int x = 0, y = 0, leaf = 0;
      bool traced = false;
      if (slot_xy(g, K, J, slot, x, y, leaf)) {
        const size_t idx = (size_t)y * g.W + x;
        traced = MODE == 0 || r.valid == nullptr || glb(r.valid)[idx] != 0;
        if (MODE == 2 && traced && glb(it.occ)[idx]) traced = false;
        sh.sRo[slot] = make_float4(glb(r.ox)[idx], glb(r.oy)[idx], glb(r.oz)[idx],
                                   glb(r.tmin)[idx]);
        sh.sRd[slot] = make_float4(glb(r.dx)[idx], glb(r.dy)[idx], glb(r.dz)[idx],
                                   glb(r.tmax)[idx]);
      }
      sh.sRv[slot] = traced ? 1 : 0;
      if (MODE != 2) sh.sKey[slot] = kMissKey;
      if (MODE == 2) sh.sAux[slot] = 0u;
      const uint64_t bal = __ballot(traced);
      if (__lane_id() == 0 && bal) atomicAdd(&sh.sTraced, __popcll(bal));
    }
    __syncthreads();
    if (sh.sV[0] && sh.sTraced > 0) {
      // The unit's clusters of frontier roots passed the cluster bound against the block
      // root.  Four clusters (256 roots) at a time: the roots that pass their own bound seed
      // the traversal stack, which is drained before the next four.  Pairs are tested when
      // their queue could not take another round's emissions, and at the end.
      const auto cl = glb(it.clist) + (size_t)b * it.nclusters + unit.z;
      const int ncl = (int)unit.w;
      bool stop = false;
      for (int k0 = 0; k0 < ncl && !stop; k0 += kThreads / kCluster) {
        if (sh.sPq > kPairCap - kThreads) {
          bvh_leaf_rays<MODE, NODE, RBMAX, LMAX>(g, it, sh);
          if (MODE == 2 && sh.sOccluded >= sh.sTraced) break;
        }
        const int k = k0 + tid / kCluster;
        const uint32_t ri = k < ncl ? cl[k] * kCluster + (uint32_t)(tid % kCluster) : it.nroots;
        if (ri < it.nroots) {
          const uint32_t node = glb(it.roots)[ri];
          V3 bmin, bmax;
          uint32_t off, np;
          bvh_box(glb(it.bvh), node, bmin, bmax, off, np);
          if (bvh_live<NODE>(off, np) && bvh_bound<NODE>(sh.sN[0], bmin, bmax)) {
            if (top == 0 && np > 0) {
              bvh_emit<MODE>(sh, node, off, np, 0, it.flags);
            } else {
              const int slot = atomicAdd(&sh.sTq, 1);
              sh.sT[slot] = node << 7;  // at most 256 seeds on an empty stack
            }
          }
        }
        __syncthreads();
        for (;;) {
          const int q = min(sh.sTq, kBvhQCap);
          if (sh.sPq > kPairCap - kThreads) {
            bvh_leaf_rays<MODE, NODE, RBMAX, LMAX>(g, it, sh);
            if (MODE == 2 && sh.sOccluded >= sh.sTraced) {
              stop = true;
              break;
            }
          }
          if (q == 0) break;
          // pop the newest items (bounded stack), room for 8 children each
          int npop = min(kBvhPop, q);
          while (npop > 0 && q - npop + 8 * npop > kBvhQCap) --npop;
          if (npop == 0) {  // cannot happen for subtrees of depth <= 12 (checked on the host)
            if (tid == 0) atomicOr(it.flags, RT_FLAG_BVH_STACK);  // reported by rt_ctx_check
            break;
          }
          uint32_t item = 0;
          const int pi = tid >> 3, c = tid & 7;
          if (pi < npop) item = sh.sT[q - npop + pi];
          __syncthreads();
          if (tid == 0) sh.sTq = q - npop;
          __syncthreads();
          bool push = false;
          uint32_t child = 0;
          if (pi < npop) {
            const uint32_t B = item >> 7;
            const int R = (int)(item & 127u);
            const int sl = sub_level(R);
            V3 bmin, bmax;
            uint32_t off, np;
            bvh_box(glb(it.bvh), B, bmin, bmax, off, np);
            const bool bleaf = np > 0, rleaf = sl == top;
            int rc = -1;
            uint32_t bc = B;
            if (!rleaf && !bleaf) {
              rc = c >> 1;
              bc = off + (uint32_t)(c & 1);
            } else if (!rleaf) {
              rc = c < 4 ? c : -2;
            } else if (!bleaf) {
              rc = c < 2 ? -1 : -2;
              bc = off + (uint32_t)c;
            } else {
              rc = -2;  // leaf x leaf items are emitted, never queued
            }
            if (rc != -2) {
              int Rn = R;
              if (rc >= 0) {
                const int pl = R - pow4_off(sl), pnl = 1 << sl;
                const int dk = pl & (pnl - 1), dj = pl >> sl;
                Rn = pow4_off(sl + 1) + (2 * dj + (rc >> 1)) * (2 * pnl) + 2 * dk + (rc & 1);
              }
              if (sh.sV[Rn]) {
                V3 cmin, cmax;
                uint32_t coff, cnp;
                bvh_box(glb(it.bvh), bc, cmin, cmax, coff, cnp);
                if (bvh_live<NODE>(coff, cnp) && bvh_bound<NODE>(sh.sN[Rn], cmin, cmax)) {
                  if (sub_level(Rn) == top && cnp > 0)
                    bvh_emit<MODE>(sh, bc, coff, cnp, Rn - pow4_off(top), it.flags);
                  else {
                    push = true;
                    child = (bc << 7) | (uint32_t)Rn;
                  }
                }
              }
            }
          }
          ballot_append(sh.sT, &sh.sTq, push, child);
          __syncthreads();
        }
        if (tid == 0) sh.sTq = 0;  // drained, or abandoned once every ray is occluded
        __syncthreads();
      }
      if (sh.sPq > 0 && !(MODE == 2 && sh.sOccluded >= sh.sTraced))
        bvh_leaf_rays<MODE, NODE, RBMAX, LMAX>(g, it, sh);
    }
    __syncthreads();
    for (int slot = tid; slot < g.rb; slot += kThreads) {
      int x, y, leaf;
      if (!slot_xy(g, K, J, slot, x, y, leaf)) continue;
      const size_t idx = (size_t)y * g.W + x;
      if (MODE == 2) {
        if (sh.sAux[slot]) glb(it.occ)[idx] = 1;
      } else {
        const unsigned long long key = sh.sKey[slot];
        if (key != kMissKey) atomicMin((unsigned long long*)&it.keys[idx], key);
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------
// Hit record: id, t, (u, v) and optionally dpdu/dpdv of computeDpTuTv.cl:8-91.
// Hit record of ray i (computeDpTuTv.cl:8-91).  naive_rule: the naive kernels' inline copy of
// that code takes the coordinate-system fallback for |det| < EPS (naive.cl:60-61,153-154)
// where computeDpTuTv.cl:57 takes it for det == 0 only.  find_t: t is the strict test's, not given.
__device__ void write_hit(const RaysDev& r, const float* __restrict__ v9,
                          const float* __restrict__ uv6, size_t i, int32_t id, float t,
                          const HitOut& out, bool naive_rule = false,
                          bool find_t = false) {
  if (id < 0) {
    out.id[i] = -1;
    out.t[i] = __int_as_float(0x7f800000);
    out.u[i] = 0.f;
    out.v[i] = 0.f;
    if (out.dpdu)
      for (int c = 0; c < 3; ++c) out.dpdu[3 * i + c] = 0.f;
    if (out.dpdv)
      for (int c = 0; c < 3; ++c) out.dpdv[3 * i + c] = 0.f;
    return;
  }
  const Tri T = load_tri(v9, (uint32_t)id);
  const V3 o = {r.ox[i], r.oy[i], r.oz[i]};
  const V3 d = {r.dx[i], r.dy[i], r.dz[i]};
  float b1, b2;
  if (find_t && mt_strict(o, d, T, t, b1, b2)) t = fkey_inv((uint32_t)(hit_key(t, id) >> 32));
  bary(o, d, T, b1, b2);
  float uv[6] = {0.f, 0.f, 1.f, 0.f, 1.f, 1.f};
  if (uv6)
    for (int k = 0; k < 6; ++k) uv[k] = uv6[6 * (size_t)id + k];
  const float b0 = 1 - b1 - b2;
  out.id[i] = id;
  out.t[i] = t;
  out.u[i] = (b0 * uv[0] + b1 * uv[2]) + b2 * uv[4];
  out.v[i] = (b0 * uv[1] + b1 * uv[3]) + b2 * uv[5];
  if (out.dpdu || out.dpdv) {
    const float du1 = uv[0] - uv[4], du2 = uv[2] - uv[4];
    const float dv1 = uv[1] - uv[5], dv2 = uv[3] - uv[5];
    const V3 dp1 = sub(T.v1, T.v3), dp2 = sub(T.v2, T.v3);
    const float det = du1 * dv2 - dv1 * du2;
    V3 pu, pv;
    if (naive_rule ? (det > -kEps && det < kEps) : det == 0.f) {
      const V3 tn = normalize(cross(T.e2, T.e1));
      if (fabsf(tn.x) > fabsf(tn.y)) {
        const float il = 1.0f / sqrtf(tn.x * tn.x + tn.z * tn.z);
        pu = {-tn.z * il, 0.f, tn.x * il};
      } else {
        const float il = 1.0f / sqrtf(tn.y * tn.y + tn.z * tn.z);
        pu = {0.f, tn.z * il, -tn.y * il};
      }
      pv = cross(tn, pu);
    } else {
      const float id2 = 1.f / det;
      pu = {(dv2 * dp1.x - dv1 * dp2.x) * id2, (dv2 * dp1.y - dv1 * dp2.y) * id2,
            (dv2 * dp1.z - dv1 * dp2.z) * id2};
      pv = {(-du2 * dp1.x + du1 * dp2.x) * id2, (-du2 * dp1.y + du1 * dp2.y) * id2,
            (-du2 * dp1.z + du1 * dp2.z) * id2};
    }
    if (out.dpdu) {
      out.dpdu[3 * i] = pu.x; out.dpdu[3 * i + 1] = pu.y; out.dpdu[3 * i + 2] = pu.z;
    }
    if (out.dpdv) {
      out.dpdv[3 * i] = pv.x; out.dpdv[3 * i + 1] = pv.y; out.dpdv[3 * i + 2] = pv.z;
    }
  }
}

// ---------------------------------------------------------------------------------------
// Per-ray path (every block, or those the cluster pass queued).  A ray's result is the argmin
// over the triangles that pass its strict leaf test AND the exact cull chain of its leaf (for
// ray-bvh: that are tested at a (BVH leaf, hierarchy leaf) pair whose lockstep chain passes).
// Every such triangle passes the strict leaf test, so each ray walks the scene's search BVH
// (padded, conservative boxes), runs the strict leaf test on the triangles of the leaves it
// reaches, and evaluates the exact chain only for those that pass it and could change the
// ray.  The (t, id) key, the repair-region key and the occlusion flag are the block path's,
// so the outcome is the same; every ray of a block is handled by exactly one lane, which
// writes its results directly.
// Hierarchy node of level l above image position (x, y), from the job's node array.  The
// job (and so g) may differ between the lanes of a wavefront: the level's table entries are
// read with the lane's own index, two loads instead of a select over every level.
template <class P>
__device__ __forceinline__ bool chain_node(const RHGeom& g, P nodes, int x, int y, int l, Node& n) {
  const int gw = g.gw[l], off = g.off[l];
  const int cxl = g.cx << l, cyl = g.cy << l;
  const P p = nodes + 4 * ((size_t)off + (size_t)(y / cyl) * gw + (x / cxl));
  const float4 a = ld4(p, 0), b = ld4(p, 1), c = ld4(p, 2), d = ld4(p, 3);
  n.dmin = {a.x, a.y, a.z};
  n.dmax = {b.x, b.y, b.z};
  n.omin = {c.x, c.y, c.z};
  n.omax = {d.x, d.y, d.z};
  return a.w != 0.f;
}

// rayhierarchy: the exact cull chain of the ray's leaf for triangle `id`
// (intersection6DB.cl:51-119 and variants: every level from the block root to the leaf).
template <int MODE, int NODE>
__device__ __forceinline__ bool ray_chain_rh(const RhItem& it, int x, int y, uint32_t id) {
  const Tri T = load_tri(glb(it.v9), id);
  for (int l = it.g.L - 1; l >= 0; --l) {
    Node n;
    if (!chain_node(it.g, glb(it.nodes), x, y, l, n)) return false;
    if (!cull_exact<MODE, NODE>(n, T)) return false;
  }
  return true;
}

// ray-bvh: the exact lockstep chain of (BVH leaf b, the ray's hierarchy leaf): step s visits
// the hierarchy node of level max(top - s, 0) and the BVH node of depth min(s, d) above b.
template <int NODE>
__device__ __forceinline__ bool ray_chain_bvh(const RhItem& it, int x, int y, uint32_t b) {
  const int top = it.g.L - 1;
  const int d = (int)glb(it.bvh_depth)[b];
  uint32_t node = b;
  int dn = d;
  for (int st = max(top, d); st >= 0; --st) {
    const int bd = min(st, d);
    while (dn > bd) {
      node = glb(it.bvh_parent)[node];
      --dn;
    }
    Node n;
    if (!chain_node(it.g, glb(it.nodes), x, y, top - min(st, top), n)) return false;
    V3 bmin, bmax;
    uint32_t off, np;
    bvh_box(glb(it.bvh), node, bmin, bmax, off, np);
    if (!bvh_live<NODE>(off, np) || !bvh_cull<NODE>(n, bmin, bmax)) return false;
  }
  return true;
}

// ---------------------------------------------------------------------------------------
// Grazing pass.  The per-ray path's tree does not find every strict hit of a ray that runs close
// to a triangle's plane (rt_search.h).  For coherent blocks, where one plane can hold many rays
// (a wall seen edge on, a light in the plane of a wall), a work-group therefore looks for the
// triangles that a ray of the block may graze and tests them directly:
//   - clusters are bounded against the block root as the cluster pass does (what the reference
//     cannot reach through its cull chain is left out), 64 of them at a time by their common box
//     first, and by the range of their triangles' planes;
//   - the triangles of the clusters left are asked whether any ray of the block may graze them:
//     by their angle, 16 bytes a triangle, and those left, compacted, by the distance of their
//     plane and their place, with intervals over the block's origins, far ends and directions
//     (camera rays have one origin, shadow rays toward a light nearly one far end), and bounded
//     against the block root themselves;
//   - every ray asks for its own angle (in a long list, every 16 rays all the questions first),
//     and takes the strict test of what is left and then the exact cull chain.
// A block whose rays lie far apart (the horizon of a ground plane) lists many triangles that
// hardly any of its rays can graze, and the launch lasted as long as it: one work-group gives such
// a block up and queues it, and a second launch takes it by kGrazeSlices work-groups, each with
// its share of the clusters.
// Hits found here are verified; they go into the ray's seed (closest) or its flag (occlusion),
// and the per-ray kernel starts from them.
// The build marks the blocks to look at (gblock 1): not incoherent ones (kIncoherent), whose
// intervals exclude nothing, unless the scene is tiny (kGrazeAll), nor blocks of more than kMaxBlockRays rays or kUnitLevels levels.
// Occlusion blocks whose root passes many clusters of a large scene (kHeavy) are left out here.
constexpr int kGrazeSecond = 1024;  // work-groups of the second launch
constexpr int kGrazeGrid = 4096;    // work-groups at most; each takes every kGrazeGrid-th block
constexpr int kGrazeAhead = 2;      // chunks of 64 records loaded at a time
constexpr int kGrazeRound = 128;    // records that a wavefront lists by angle before the next step
constexpr int kGrazeBatch = 128;    // listed triangles tested at a time
constexpr int kGrazeFew = 48;       // the length of a long list
constexpr int kGrazeSlices = 16;    // work-groups to a queued block
constexpr uint32_t kGrazeAll = 128;  // triangles that every ray can test: incoherent blocks too
constexpr uint32_t kGrazeMany = 192;  // listed triangles that queue a block
template <int WAVES>
struct GrazeShared {
  static constexpr int kNear = WAVES * (kGrazeRound + 64 * kGrazeAhead);
  static constexpr int kList = 512 + kNear;
  float box[kMaxBlockRays / 16][20];  // per 16 rays: ends of origin, far end, direction; dmin
  GrazeRays rays[kMaxBlockRays / 16];
  GrazeRays all;
  uint32_t near[kNear];            // records that pass by their angle
  uint32_t tri[kList];             // records that pass for the block
  // the batch at hand: GrazeNormal, RhItem::gtest, and in a long list GrazeTri
  float4 N[kGrazeBatch], T[kGrazeBatch][3], G[kGrazeBatch][3];
  int nnear, ntri, any, passed, marked;
};

// A ray's seed: its key, bit 31 inverted when a repair-region hit lies at exactly tmin.
__device__ __forceinline__ uint64_t seed_pack(uint64_t key, bool mark) {
  return key ^ (mark ? 0x80000000ull : 0ull);
}
__device__ __forceinline__ void seed_unpack(uint64_t s, uint64_t& key, bool& mark) {
  mark = ((s >> 31) & 1u) != ((uint32_t)(s >> 32) == 0xffffffffu ? 1u : 0u);
  key = seed_pack(s, mark);
}
template <int M>
__device__ __forceinline__ float min_group(float v) {
  return fminf(v, __int_as_float(from_group<M>(__float_as_int(v))));
}
__device__ __forceinline__ float min_row(float v) {  // over the 16 lanes of a row
  return min_group<8>(min_group<4>(min_group<2>(min_group<1>(v))));
}
__device__ __forceinline__ GrazeTri load_graze(const GrazeTri* p, size_t i) {
  const auto q = (RT_GLOBAL const float4*)p;
  const float4 a = ld4(q, 3 * i), b = ld4(q, 3 * i + 1), c = ld4(q, 3 * i + 2);
  return GrazeTri{{a.x, a.y, a.z}, a.w, b.x, b.y, __float_as_uint(b.z), b.w, {c.x, c.y, c.z}, c.w};
}

template <int MODE, int NODE, bool BVH, int WAVES>
__device__ __forceinline__ bool graze_block(const RhItem& it, int b, int slice, int slices,
                                            GrazeShared<WAVES>& sh) {
  constexpr int kWork = 64 * WAVES;
  const uint32_t mates = (uint32_t)(WAVES * slices);  // wavefronts at the block
  const RHGeom& g = it.g;
  const RaysDev& r = it.r;
  const SearchFrame frame = it.sframe;
  const float4 *const cbox = it.cbox, *const gbox = it.gbox;
  const GrazeCluster* const gcluster = it.gcluster;
  const GrazeNormal* const gnormal = it.gnormal;
  const uint32_t* const gfirst = it.gfirst;
  const uint32_t ntri = it.ntri;
  const float inf = __int_as_float(0x7f800000);
  const int tid = threadIdx.x, lane = __lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int top = g.L - 1;
  const int K = b % g.gw[top], J = b / g.gw[top];
  const int rows = (g.rb + 15) / 16;
  if (tid == 0) sh.nnear = sh.ntri = sh.any = sh.passed = sh.marked = 0;
  // the boxes of every 16 rays, lower ends and negated upper ends
#pragma unroll 1
  for (int s0 = wave * 64; s0 < g.rb; s0 += kWork) {
    float v[19];
    int x = 0, y = 0, leaf = 0;
    bool in = slot_xy(g, K, J, s0 + lane, x, y, leaf);
    const size_t i = in ? (size_t)y * g.W + x : 0;
    const V3 o = {glb(r.ox)[i], glb(r.oy)[i], glb(r.oz)[i]};
    const V3 d = {glb(r.dx)[i], glb(r.dy)[i], glb(r.dz)[i]};
    const float tm = glb(r.tmax)[i], s = tm < inf ? tm : 1.f;
    if (MODE != 0 && r.valid != nullptr) in = in && glb(r.valid)[i] != 0;
    // a ray that is not finite passes no test
    in = in && fabsf(o.x) < inf && fabsf(o.y) < inf && fabsf(o.z) < inf && fabsf(d.x) < inf &&
         fabsf(d.y) < inf && fabsf(d.z) < inf;
    const float p[9] = {o.x, o.y, o.z, o.x + s * d.x, o.y + s * d.y, o.z + s * d.z,
                        d.x, d.y, d.z};
    for (int c = 0; c < 9; ++c) {
      v[6 * (c / 3) + c % 3] = in ? p[c] : inf;
      v[6 * (c / 3) + 3 + c % 3] = in ? -p[c] : inf;
    }
    v[18] = in ? fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z)) : inf;
    for (int c = 0; c < 19; ++c) v[c] = min_row(v[c]);
    if ((lane & 15) == 0)
      for (int c = 0; c < 19; ++c) sh.box[(s0 + lane) / 16][c] = v[c];
  }
  __syncthreads();
  auto rays_of = [&](const float* v) {
    float hi[9];
    for (int c = 0; c < 9; ++c) hi[c] = -v[6 * (c / 3) + 3 + c % 3];
    return graze_rays(v, hi, v + 6, hi + 3, v + 12, hi + 6, v[18], frame);
  };
  if (wave == 0) {
    float m = inf, v[19];
    if (lane < 19)
      for (int q = 0; q < rows; ++q) m = fminf(m, sh.box[q][lane]);
    for (int c = 0; c < 19; ++c)
      v[c] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), c));
    const GrazeRays a = rays_of(v);
    if (lane == 0) sh.all = a;
  }
  const RT_GLOBAL float4* const p =
      glb(it.nodes) + 4 * ((size_t)g.off[top] + (size_t)J * g.gw[top] + K);
  Node root;
  {
    const float4 a0 = ld4(p, 0), a1 = ld4(p, 1), a2 = ld4(p, 2), a3 = ld4(p, 3);
    root.dmin = {a0.x, a0.y, a0.z};
    root.dmax = {a1.x, a1.y, a1.z};
    root.omin = {a2.x, a2.y, a2.z};
    root.omax = {a3.x, a3.y, a3.z};
  }
  __syncthreads();
  GrazeRays all = sh.all;
  {  // uniform: to scalar registers
    auto scalar = [](float& q) { q = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(q))); };
    for (F3* q : {&all.oc, &all.oh, &all.qc, &all.qh, &all.dc, &all.dh}) {
      scalar(q->x);
      scalar(q->y);
      scalar(q->z);
    }
    for (float* q : {&all.dist, &all.far, &all.dir, &all.extra}) scalar(*q);
    all.all = __builtin_amdgcn_readfirstlane((int)all.all) != 0;
    for (V3* q : {&root.dmin, &root.dmax, &root.omin, &root.omax}) {
      scalar(q->x);
      scalar(q->y);
      scalar(q->z);
    }
  }
  // what a record's slope is multiplied by (GrazeNormal)
  const float steep = graze_steep(all, frame);
  auto box_passes = [&](const float4* box, uint32_t k) {
    const float4 lo = ld4(glb(box), 2 * (size_t)k), hi = ld4(glb(box), 2 * (size_t)k + 1);
    return cluster_bound<MODE, NODE, BVH>(root, V3{lo.x, lo.y, lo.z}, V3{hi.x, hi.y, hi.z});
  };
  // The same for one triangle.  ray-bvh: its reference BVH leaf meets the ray's hierarchy leaf,
  // not the root; a cluster's bound over the root's rays holds for every node below it if its
  // box covers the roundings of their centres and half widths.
  auto root_passes = [&](uint32_t id) {
    const Tri T = load_tri(glb(it.v9), id);
    if constexpr (!BVH) {
      return cull_bound<MODE, NODE>(root, T);
    } else {
      const uint32_t leaf = glb(it.tleaf)[id];
      if (leaf == 0xffffffffu) return false;
      V3 mn, mx;
      uint32_t off, np;
      bvh_box(glb(it.bvh), leaf & 0x7fffffffu, mn, mx, off, np);
      if constexpr (NODE != 1) {
        auto slack = [](float a0, float a1, float c0, float c1) {
          return 0x1p-20f * (fmaxf(fabsf(a0), fabsf(a1)) + fmaxf(fabsf(c0), fabsf(c1)));
        };
        const V3 w = {slack(mn.x, mx.x, root.omin.x, root.omax.x),
                      slack(mn.y, mx.y, root.omin.y, root.omax.y),
                      slack(mn.z, mx.z, root.omin.z, root.omax.z)};
        mn = sub(mn, w);
        mx = add(mx, w);
      }
      return cluster_bound<MODE, NODE, BVH>(root, mn, mx);
    }
  };
  // the wavefront's share of the clusters: one in `mates` of the groups of 64 that pass, or in
  // small scenes of the clusters
  const uint32_t nclusters = it.nclusters, ngroups = (nclusters + 63u) / 64u;
  const uint32_t mate = (uint32_t)(slice * WAVES + wave);
  const bool by_cluster = ngroups <= mates / 2;
  uint32_t gbase = 0, group = 0, turn = 0, pos = 0, end = 0;
  uint64_t gmask = 0, cmask = 0;
  bool fresh = true;
  // whether enough clusters pass decides first: a round that only counts
  const uint32_t enough = BVH ? kHeavyBvh : kHeavy;
  bool count = MODE == 2 && slices == 1 && nclusters >= 4u * enough;
  int passed = 0;
  auto next_chunk = [&]() {  // up to 64 records from pos
#pragma unroll 1
    for (;;) {
      if (pos < end) return true;
      if (cmask != 0) {
        const uint32_t c = group * 64u + (uint32_t)__ffsll((unsigned long long)cmask) - 1u;
        cmask &= cmask - 1;
        if (by_cluster && turn++ % mates != mate) continue;
        pos = gfirst ? glb(gfirst)[c] : c * (uint32_t)kCluster;
        end = gfirst ? glb(gfirst)[c + 1]
                        : min(c * (uint32_t)kCluster + (uint32_t)kCluster, ntri);
        continue;
      }
      // the next group of clusters that passes, or (gmask empty) the next 64 groups
      const bool inner = gmask != 0;
      if (inner) {
        group = gbase + (uint32_t)__ffsll((unsigned long long)gmask) - 1u;
        gmask &= gmask - 1;
        if (!by_cluster && turn++ % mates != mate) continue;
      } else {
        gbase = fresh ? 0u : gbase + 64u;
        fresh = false;
        if (gbase >= ngroups) return false;
        if (ngroups == 1u) {  // its clusters say as much
          gmask = 1u;
          continue;
        }
      }
      const uint32_t q = (inner ? group * 64u : gbase) + (uint32_t)lane;
      const bool exists = q < (inner ? nclusters : ngroups);
      float4 a0{}, a1{}, a2{};
      if (exists && inner) {
        const auto w = (RT_GLOBAL const float4*)gcluster;
        a0 = ld4(w, 3 * (size_t)q);
        a1 = ld4(w, 3 * (size_t)q + 1);
        a2 = ld4(w, 3 * (size_t)q + 2);
      }
      const bool ok = exists && box_passes(inner ? cbox : gbox, q);
      if (!inner) {
        gmask = __ballot(ok);
        continue;
      }
      if (count) {
        passed += __popcll(__ballot(ok));
        continue;
      }
      cmask = __ballot(ok && grazes_cluster(all, GrazeCluster{{a0.x, a0.y, a0.z}, a0.w,
                                                              {a1.x, a1.y, a1.z}, a1.w, a2.x,
                                                              a2.y, a2.z, 0.f}, frame));
    }
  };
  bool first = true;
  // the rays' tests against the listed triangles; empties the list
  auto flush = [&]() {
    const int n = sh.ntri;
    const bool ask = n > kGrazeFew;
    if (ask && tid < rows) sh.rays[tid] = rays_of(sh.box[tid]);
    const bool init = first && slices == 1;
    first = false;
#pragma unroll 1
    for (int base = 0; base < n; base += kGrazeBatch) {
      const int m = min(n - base, kGrazeBatch);
      for (int e = tid; e < 4 * m; e += kWork) {
        const size_t rec = sh.tri[base + (e >> 2)];
        if ((e & 3) == 3) sh.N[e >> 2] = ld4((RT_GLOBAL const float4*)gnormal, rec);
        else sh.T[e >> 2][e & 3] = ld4((RT_GLOBAL const float4*)it.gtest, 3 * rec + (e & 3));
        if (ask && (e & 3) != 3)
          sh.G[e >> 2][e & 3] = ld4((RT_GLOBAL const float4*)it.graze, 3 * rec + (e & 3));
      }
      __syncthreads();
      // 16 rays at a time, four lanes a ray
#pragma unroll 1
      for (int row = wave; row < rows; row += WAVES) {
        const int slot = row * 16 + (lane & 15), sub = lane >> 4;
        int x = 0, y = 0, hleaf = 0;
        bool alive = slot_xy(g, K, J, slot, x, y, hleaf);
        const size_t i = alive ? (size_t)y * g.W + x : 0;
        const V3 o = {glb(r.ox)[i], glb(r.oy)[i], glb(r.oz)[i]};
        const V3 d = {glb(r.dx)[i], glb(r.dy)[i], glb(r.dz)[i]};
        const float tmin = glb(r.tmin)[i], tmax = MODE == 2 ? glb(r.tmax)[i] : inf;
        if (MODE != 0 && r.valid != nullptr) alive = alive && glb(r.valid)[i] != 0;
        const bool fresh_ray = init && base == 0;
        uint64_t best = kMissKey;
        bool mark = false, found = false;
        if (alive && !fresh_ray) {
          if (MODE == 2) found = glb(it.occ)[i] != 0;
          else if (slices > 1) best = __hip_atomic_load(&it.gseed[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          else seed_unpack(glb(it.gseed)[i], best, mark);
        }
        const uint64_t best0 = best;
        float len, dist;
        graze_ray(F3{o.x, o.y, o.z}, F3{d.x, d.y, d.z}, frame, len, dist);
#pragma unroll 1
        for (int e0 = 0; e0 < m; e0 += 64) {
          const int k = min(m - e0, 64);
          uint64_t todo = k < 64 ? (1ull << k) - 1ull : ~0ull;
          if (ask) {
            bool ok = false;
            if (lane < k) {
              const float4 a = sh.G[e0 + lane][0], c1 = sh.G[e0 + lane][1], c2 = sh.G[e0 + lane][2];
              ok = grazes(sh.rays[row],
                          GrazeTri{{a.x, a.y, a.z}, a.w, c1.x, c1.y, __float_as_uint(c1.z), c1.w,
                                   {c2.x, c2.y, c2.z}, c2.w}, frame);
            }
            todo &= __ballot(ok);
          }
          todo &= 0x1111111111111111ull << sub;
          if (!alive || (MODE == 2 && found)) todo = 0;
          // lanes go on to their next hit, whose chains are then evaluated together
#pragma unroll 1
          while (__any(todo != 0)) {
            uint32_t id = 0, leaf = 0;
            uint64_t key = kMissKey;
            bool um = false, rp = false;
#pragma unroll 1
            for (; todo != 0 && !um && !rp; todo &= todo - 1) {
              const int j = e0 + __ffsll((unsigned long long)todo) - 1;
              const float4 q = sh.N[j], tc = sh.T[j][2];
              // the ray's own angle
              if (graze_clears(GrazeNormal{{q.x, q.y, q.z}, q.w}, tc.w, F3{d.x, d.y, d.z}, len,
                               dist))
                continue;
              const float4 ta = sh.T[j][0], tb = sh.T[j][1];
              Tri S;
              S.v1 = {ta.x, ta.y, ta.z};
              S.e1 = {ta.w, tb.x, tb.y};
              S.e2 = {tb.z, tb.w, tc.x};
              S.v2 = S.v3 = S.v1;
              float t, b1, b2;
              if (!mt_strict(o, d, S, t, b1, b2)) continue;
              id = __float_as_uint(tc.y);
              leaf = __float_as_uint(tc.z);
              // in no leaf; or not its leaf's first primitive (6DB / IA secondary rays)
              if (BVH && (leaf == 0xffffffffu ||
                          (MODE == 1 && NODE != 2 && (leaf & 0x80000000u))))
                continue;
              key = hit_key(t, (int32_t)id);
              um = t > tmin && t < tmax && (MODE == 2 || key < best);
              rp = MODE == 0 && !BVH && it.repair_run > 0 && !mark && repair_kept(t, tmin) &&
                   repair_region(b1, b2);
            }
            bool ok = um || rp;
            if (ok) {
              // most that fail do so in the ray's leaf, which its bound tells for less
              Node nd;
              ok = chain_node(it.g, glb(it.nodes), x, y, 0, nd);
              if constexpr (BVH) {
                V3 mn, mx;
                uint32_t off, np;
                bvh_box(glb(it.bvh), leaf & 0x7fffffffu, mn, mx, off, np);
                ok = ok && bvh_bound<NODE>(nd, mn, mx) &&
                     ray_chain_bvh<NODE>(it, x, y, leaf & 0x7fffffffu);
              } else {
                ok = ok && cull_bound<MODE, NODE>(nd, load_tri(glb(it.v9), id)) &&
                     ray_chain_rh<MODE, NODE>(it, x, y, id);
              }
            }
            if (!ok) continue;
            found = true;
            if (MODE == 2) todo = 0;
            if (um) best = key;
            if (rp) mark = true;
          }
        }
        // the four lanes' results together
        for (int c = 16; c < 64; c <<= 1) {
          const uint64_t q = ((uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)(best >> 32), c) << 32) |
                             (uint32_t)__shfl_xor((int)(uint32_t)best, c);
          best = q < best ? q : best;
          mark = __shfl_xor((int)mark, c) != 0 || mark;
          found = __shfl_xor((int)found, c) != 0 || found;
        }
        if (slices > 1) {  // others are at the ray too
          if (alive && sub == 0 && found) {
            if (MODE == 2) glb(it.occ)[i] = 1;
            else atomicMin((unsigned long long*)&it.gseed[i], (unsigned long long)best);
            if (mark) sh.marked = 1;
          }
        } else if (alive && sub == 0 && (found || fresh_ray)) {
          if (MODE == 2) glb(it.occ)[i] = found ? 1 : 0;
          else glb(it.gseed)[i] = seed_pack(best, mark);
        }
        if (__any(found && (MODE == 2 || best != best0 || mark)) && lane == 0) sh.any = 1;
      }
      __syncthreads();
    }
    if (tid == 0) sh.ntri = 0;
    __syncthreads();
  };
  uint32_t listed = 0, kept = 0;
  // Rounds: the wavefronts list the records of their share by angle, up to kGrazeRound and one
  // load each, and then share out the list for the other questions.
  bool done = false;
#pragma unroll 1
  for (;;) {
#pragma unroll 1
    for (int added = 0; !done && added < kGrazeRound;) {
      // chunk u's ends in lane u
      uint32_t from = 0, to = 0;
#pragma unroll 1
      for (int u = 0; u < kGrazeAhead && !done; ++u) {
        done = !next_chunk();
        if (!done && lane == u) {
          from = pos;
          to = end;
        }
        pos += 64u;
      }
      float4 q[kGrazeAhead];
      uint32_t at[kGrazeAhead];
      uint64_t m[kGrazeAhead];
      bool in[kGrazeAhead];
#pragma unroll
      for (int u = 0; u < kGrazeAhead; ++u) {
        at[u] = __builtin_amdgcn_readlane(from, u) + (uint32_t)lane;
        in[u] = at[u] < (uint32_t)__builtin_amdgcn_readlane(to, u);
        if (in[u]) q[u] = ld4((RT_GLOBAL const float4*)gnormal, at[u]);
      }
      int cnt = 0;
#pragma unroll
      for (int u = 0; u < kGrazeAhead; ++u) {
        m[u] = __ballot(in[u] && grazes_angle(all, steep, GrazeNormal{{q[u].x, q[u].y, q[u].z},
                                                                      q[u].w}));
        cnt += __popcll(m[u]);
      }
      if (cnt == 0) continue;
      int base = 0;
      if (lane == 0) base = atomicAdd(&sh.nnear, cnt);
      base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
      for (int u = 0; u < kGrazeAhead; ++u) {
        if ((m[u] >> lane) & 1u) sh.near[base + __popcll(m[u] & ((1ull << lane) - 1ull))] = at[u];
        base += __popcll(m[u]);
      }
      added += cnt;
    }
    if (count) {  // uniform; by_cluster: every wavefront has counted all of them
      if (lane == 0) atomicAdd(&sh.passed, passed);
      __syncthreads();
      if ((uint32_t)sh.passed >= enough * (by_cluster ? (uint32_t)WAVES : 1u)) break;
      count = done = false;
      fresh = true;
      turn = 0;
      continue;
    }
    const bool more = __syncthreads_or(!done) != 0;
    const int nnear = sh.nnear;
    listed += (uint32_t)nnear;
#pragma unroll 1
    for (int e = wave * 64; e < nnear; e += kWork) {
      bool ok = false;
      uint32_t k = 0;
      if (e + lane < nnear) {
        k = sh.near[e + lane];
        const GrazeTri q = load_graze(it.graze, k);
        ok = grazes(all, q, frame) && root_passes(q.id);
      }
      const uint64_t m = __ballot(ok);
      if (m == 0) continue;
      int base = 0;
      if (lane == 0) base = atomicAdd(&sh.ntri, __popcll(m));
      base = __builtin_amdgcn_readfirstlane(base);
      if (ok) sh.tri[base + __popcll(m & ((1ull << lane) - 1ull))] = k;
    }
    __syncthreads();
    if (tid == 0) sh.nnear = 0;
    if (slices == 1) {  // uniform
      kept += (uint32_t)sh.ntri;
      if (kept > kGrazeMany || listed > kGrazeMany * 16u + 64u * ngroups) {
        // to the second launch; no ray has a hit yet
        for (int slot = tid; slot < g.rb; slot += kWork) {
          int x = 0, y = 0, leaf = 0;
          if (!slot_xy(g, K, J, slot, x, y, leaf)) continue;
          const size_t i = (size_t)y * g.W + x;
          if (MODE == 2) glb(it.occ)[i] = 0;
          else glb(it.gseed)[i] = kMissKey;
        }
        if (tid == 0) glb(it.gblock)[b] = 1u;
        return false;
      }
    }
    if (sh.ntri > (more ? sh.kList - sh.kNear : 0)) flush();
    if (!more) break;
    __syncthreads();
  }
  // a repair-region hit of some ray in a slice: all rays of the block count as having one, which
  // only sends them through the repair pass
  if (tid == 0 && sh.any != 0) {
    if (slices == 1) glb(it.gblock)[b] = kGrazeHit;
    else atomicMax(&it.gblock[b], MODE == 0 && sh.marked != 0 ? kGrazeMark : kGrazeHit);
  }
  return true;
}

// heavy: the blocks queued for the second launch, their number in ctr[5].  slices: work-groups to a
// block; 1 in the first launch.  queued: only the blocks in `heavy`.
template <int MODE, int NODE, bool BVH, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(4))) void
rh_graze_kernel(const RhItem* __restrict__ items, int nitems, uint32_t nblocks,
                uint32_t* __restrict__ ctr, uint32_t* __restrict__ heavy, uint32_t slices,
                bool queued) {
  __shared__ GrazeShared<WAVES> sh;
  const uint32_t n = (queued ? __builtin_amdgcn_readfirstlane(ctr[5]) : nblocks) * slices;
  for (uint32_t i0 = 0; i0 * gridDim.x + blockIdx.x < n; i0 += 64) {
    // lane u: the work-group's block (or slice) number i0 + u
    const uint64_t at = (uint64_t)(i0 + (uint32_t)__lane_id()) * gridDim.x + blockIdx.x;
    bool look = at < n;
    if (look && !queued) {
      const uint32_t gb = (uint32_t)at / slices;
      const RhItem& it = items[find_block_item_lane(items, nitems, gb)];
      look = it.gblock != nullptr && glb(it.gblock)[gb - it.block_base] != 0u;
    }
    for (uint64_t m = __ballot(look); m != 0; m &= m - 1) {
      const uint32_t u =
          (i0 + (uint32_t)__ffsll((unsigned long long)m) - 1u) * gridDim.x + blockIdx.x;
      const uint32_t gb = queued ? __builtin_amdgcn_readfirstlane(heavy[u / slices]) : u / slices;
      const RhItem& it = items[nitems == 1 ? 0 : find_block_item(items, nitems, gb)];
      if (!graze_block<MODE, NODE, BVH, WAVES>(it, (int)(gb - it.block_base), (int)(u % slices),
                                               (int)slices, sh)) {
        if (threadIdx.x == 0) heavy[atomicAdd(&ctr[5], 1u)] = gb;
      }
      __syncthreads();
    }
  }
}

// ctr: the counters to clear for the kernels that follow (null: the init kernel does it).
template <bool USE_VALID, bool UV, bool ONE>
__device__ __forceinline__ void group_build(const RhItem& it, uint32_t* __restrict__ ctr) {
  __shared__ float sBox[kMaxSub][12];
  __shared__ int sVal[kMaxSub];
  if (ctr != nullptr && blockIdx.x == 0) clear_counters(ctr, threadIdx.x);
  const int b = (int)(blockIdx.x - it.block_base);
  if (it.g.L > kUnitLevels) {
    build_block_deep<USE_VALID, UV, ONE>(it.g, it.r, it.nodes, b);
    return;
  }
  build_block<USE_VALID, UV, ONE>(it.g, it.r, it.nodes, b, sBox, sVal);
  if (it.gblock != nullptr && threadIdx.x < 64) {
    // whether the grazing pass looks at the block: the mean direction spread of its leaves, as in
    // the cluster pass
    const int lane = threadIdx.x, nleaf = it.g.nlx * it.g.nlx;
    float sp = 0.f;
    const bool have = lane < nleaf && sVal[it.g.nsub - nleaf + lane] != 0;
    if (have) {
      const float* v = sBox[it.g.nsub - nleaf + lane];
      sp = UV ? v[4] - v[1] : fmaxf(fmaxf(v[3] - v[0], v[4] - v[1]), v[5] - v[2]);
    }
    for (int m = 32; m > 0; m >>= 1) sp += __shfl_xor(sp, m);
    const int n = __popcll(__ballot(have));
    const bool look =
        n > 0 && it.ntri > 0 && (it.ntri <= kGrazeAll || !(sp > kIncoherent * (float)n));
    if (lane == 0) glb(it.gblock)[b] = look ? 1u : 0u;
    if (look && it.gsliced) {  // no ray has a hit yet
      const int top = it.g.L - 1;
      for (int slot = lane; slot < it.g.rb; slot += 64) {
        int x = 0, y = 0, leaf = 0;
        if (!slot_xy(it.g, b % it.g.gw[top], b / it.g.gw[top], slot, x, y, leaf)) continue;
        const size_t i = (size_t)y * it.g.W + x;
        if (it.occ != nullptr) glb(it.occ)[i] = 0;
        else glb(it.gseed)[i] = kMissKey;
      }
    }
  }
}
template <bool USE_VALID, bool UV, bool ONE>
__global__ __launch_bounds__(256) void rh_group_build_kernel(const RhItem* __restrict__ items,
                                                             int nitems,
                                                             uint32_t* __restrict__ ctr) {
  group_build<USE_VALID, UV, ONE>(items[find_block_item(items, nitems, blockIdx.x)], ctr);
}
// The same for a single job whose table entry comes with the launch; the first work-group leaves
// it in `table` for the kernels that follow.  A renderer whose buffers change from call to call
// thus uploads nothing: the copy (3.5 us), its event and the wait for the one before are gone.
template <bool USE_VALID, bool UV, bool ONE>
__global__ __launch_bounds__(256) void rh_single_build_kernel(const RhItem it,
                                                              RhItem* __restrict__ table,
                                                              uint32_t* __restrict__ ctr) {
  if (blockIdx.x == 0) {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(&it);
    for (uint32_t i = threadIdx.x; i < sizeof(RhItem) / 4; i += kThreads)
      reinterpret_cast<uint32_t*>(table)[i] = src[i];
  }
  group_build<USE_VALID, UV, ONE>(it, ctr);
}

// Compare-exchange of two sort keys.
__device__ __forceinline__ void key_swap(uint32_t& a, uint32_t& b) {
  const uint32_t lo = min(a, b);
  b = max(a, b);
  a = lo;
}

// Per-ray kernel: one wavefront per work-group, every lane one ray at a time.  The queue holds
// 64-ray chunks; a wavefront takes a chunk and deals its rays to lanes without one, and when a
// lane's ray is done it takes the next ray of the chunk (or of the next chunk) at the next
// round, so lanes of long traversals do not leave the others idle.  A round walks interior
// nodes until most lanes hold a leaf or are done (Aila and Laine's while-while), then tests
// the postponed leaves.
//
// A ray is first traced as if every cull chain passed, which is what they nearly always do:
// occlusion ends at its first strict hit inside the interval, a closest hit is the nearest
// strict hit.  That one candidate goes to a wavefront queue in LDS as {ray, triangle or BVH
// leaf, job} (a closest hit's t, or its key, goes to memory) and its lane takes the next
// ray; whenever the queue holds 64 candidates, their chains are evaluated together, one per
// lane.  A passing chain confirms the candidate: the nearest strict hit is the answer when its
// chain passes, and any strict hit with a passing chain occludes.  A ray whose candidate
// failed goes to a second stack in the same LDS, from which idle lanes take it before new rays
// and trace it from the root again, evaluating each candidate's chain at once and pruning with
// verified hits only.  So does a primary ray whose nearest repair-region hit (chains aside) lies
// low enough to matter to the repair pass, which needs verified repair candidates, and a ray
// whose candidate finds the queue full.
//
// Before, each improvement of a ray's bound and every repair-region hit had its chain evaluated
// and lanes waited for theirs, a quarter of a wavefront at a time, in a launch's tail one by
// one.  Measured, every block per-ray, with rounds that walk until half of the lanes hold a leaf
// (1/8 before): torus 512 x 512 closest 247 -> 142 us, occlusion 318 -> 146; room task to path
// depth 3, the bounces' closest hits 2,816 -> 1,767, occlusion 2,278 -> 1,251; 1 M segments
// 1,089 -> 688; camera rays of twelve scenes 1,049 -> 609.
//
// Without a queue of chunks (rq null) every block of the group is traced here: chunk e is found
// from the jobs' chunk prefixes and the results are written here, misses by their lane and hits
// by the lane that confirms them, so no reduction keys, no init and no finalize launch are
// needed.  Otherwise the rays of the blocks that the cluster pass sent here leave their keys,
// repair keys and flags as the block path does.
// ONE: the group has one job; its table entry and the pointers in it are then uniform.
//
// Once the wavefront has no ray left to deal, its lanes run dry one after another while its
// longest rays go on (a chunk's longest walk is 2-3 times its mean).  From then on it splits
// rays: whenever at most kSplitLanes lanes hold one, each of those with unvisited nodes on its
// stack gives the oldest of them, with a copy of the ray, to an idle lane.  The lanes of a ray
// share its bound (or the news of its candidate) through LDS, and the last of them to finish
// decides the ray.  Measured: 1 M segments 596 -> 455 us, room task path depth 3, secondary
// 1,104 -> 813 and occlusion 953 -> 629, twelve scenes' segments 398 -> 290, 100x4 leaves closest
// 249 -> 114, box_uv clusters 164 -> 82.  Splitting from 32 busy lanes was up to 10% slower than
// from 48, from 16 up to 50%; every second round up to 20%, every fourth up to 70%.
//
// A launch of at most one chunk per resident wavefront deals each its rays at once (`spread` of
// them), in runs of 16 taken from distant parts of the launch: neighbouring rays are long
// together, and the launch lasts as long as its longest wavefront.  With whole chunks the mean
// wavefront of the torus 512 x 512 occlusion ended after 18 us, the last after 114; now 31 and
// 69 (119 -> 70 us, closest 93 -> 85; 333 x 251 ia 72 -> 53 and 69 -> 57).  Fewer rays than that
// are spread over more wavefronts, at least four each (64 wavefronts of 64 rays 44 us, 1,024 of
// 4 31 us); more wavefronts than are resident run one after another (333 x 251: 69 -> 124).
constexpr uint32_t kChainQ = 127;  // below 64 before a round, one more per lane in it
constexpr uint32_t kSplitLanes = 48;
// Idle lanes from which a wavefront deals new rays.  A deal is a chain of loads that every lane
// waits for; one for each idle lane took 18-25% of a long launch (1 M camera rays, 200,000
// triangles: any idle lane 801 us, 4 lanes 769, 8 765, 16 761, 24 781; twelve scenes 561, 523,
// 507, 499, 494).
constexpr uint32_t kDealLanes = 16;
// A word of LDS that other lanes of the wavefront change by atomics.
template <class T>
__device__ __forceinline__ T lds_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
// State of a split ray (sRay): lanes at work in bits 0..7, then a hit that the repair pass must
// see (primary, repair_kept), or the candidate found (occlusion).
constexpr uint32_t kRayLanes = 255u, kRayMark = 256u;
// Registers for four wavefronts per SIMD (128 VGPRs) and LDS for as many, see kSearchStack; with
// registers for five (96, 15-30 spilled) the room task's secondary rays took 1,315 us, the torus
// closest hits 134 us (94).  Keeping only 24 or 16 stack entries in LDS and the rest in scratch
// memory, for more work-groups per CU, was 3-6% slower.
template <int MODE, int NODE, bool BVH, bool ONE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void ray_path_kernel(
    const RhItem* __restrict__ items, int nitems, const uint2* __restrict__ rq,
    uint32_t* __restrict__ ctr, uint32_t* __restrict__ replist, uint32_t nchunks, uint32_t spread,
    uint32_t walk64) {
  __shared__ uint32_t sStk[kSearchStack][64];
  // candidates [0, qn) and, from the far end, rays to trace again [kChainQ - nf, kChainQ)
  __shared__ uint32_t sQIdx[kChainQ], sQRef[kChainQ];
  __shared__ uint16_t sQJob[kChainQ];
  __shared__ unsigned long long sBest[MODE == 2 ? 1 : 64];  // split rays, by the lane that had it
  __shared__ uint32_t sRay[64];
  constexpr uint32_t kDone = 0xffffffffu;  // not a reference (positions are below 2^31)
  const float kInf = __int_as_float(0x7f800000);
  auto widened = [](float t) { return t + fabsf(t) * kSlack; };
  const int lane = threadIdx.x;
  const uint64_t lanes_below = (1ull << lane) - 1ull;
  // wavefront-uniform: the chunk being dealt and its next slot, the queue's counts
  uint32_t cjob = 0, cblk = 0, cpart = 0, cslot = 64;
  uint32_t qn = 0, nf = 0;
  bool more = true, split = false;
  // lane state
  bool act = false, careful = false;
  uint32_t jk = 0, idx = 0;
  V3 o = {0.f, 0.f, 0.f}, d = {0.f, 0.f, 1.f};
  SlabRay sr{};
  // tlo, thi: the interval's ends, widened; thi follows the closest bound
  float tmin = 0.f, tmax = 0.f, tlo = 0.f, thi = 0.f;
  uint64_t best = kMissKey;   // closest: the nearest hit (verified when careful)
  bool mark = false;          // primary: a repair-region hit kept apart (likewise)
  uint32_t cand = 0;          // occlusion: the candidate triangle, for ray-bvh its BVH leaf
  bool track_rep = false;
  int sp = 0, sb = 0;         // the lane's stack entries [sb, sp)
  uint32_t own = 0;           // the lane whose sRay / sBest a split ray uses
  uint32_t cur = kDone, pl = kDone;
  auto pop = [&]() { return sp > sb ? sStk[--sp][lane] : kDone; };
  const bool direct = rq == nullptr;
  // the cluster pass sets ctr[4] when it routed any block here
  if (!direct && __builtin_amdgcn_readfirstlane(ctr[4]) == 0u) return;
  UnitClaim claim = claim_start();
  auto item = [&](uint32_t j) -> const RhItem& { return items[ONE ? 0u : j]; };
  // the exact chain of ray ri's candidate: a triangle, or for ray-bvh occlusion its BVH leaf
  auto chain = [&](const RhItem& it, uint32_t ri, uint32_t ref) {
    const int x = (int)(ri % (uint32_t)it.g.W), y = (int)(ri / (uint32_t)it.g.W);
    if constexpr (BVH)
      return ray_chain_bvh<NODE>(it, x, y, MODE == 2 ? ref : glb(it.tleaf)[ref] & 0x7fffffffu);
    else
      return ray_chain_rh<MODE, NODE>(it, x, y, ref);
  };
  // direct: the record of a ray that hits nothing / has hit triangle id
  auto write_miss = [&](const RhItem& it, uint32_t ri) {
    if constexpr (MODE == 2) glb(it.occ)[ri] = 0;
    else write_hit(it.r, it.v9, it.uv6, ri, -1, 0.f, it.out);
  };
  auto restart = [&]() {
    careful = true;
    best = kMissKey;
    mark = false;
    if constexpr (MODE != 2) {  // the grazing pass's hit, which is verified
      const RhItem& it = item(jk);
      if (it.gblock != nullptr) {
        const RHGeom& g = it.g;
        const uint32_t y = idx / (uint32_t)g.W, x = idx - y * (uint32_t)g.W;
        const uint32_t blk = y / (uint32_t)g.bh * (uint32_t)g.gw[g.L - 1] + x / (uint32_t)g.bw;
        const uint32_t hit = glb(it.gblock)[blk];
        if (hit == kGrazeHit) seed_unpack(glb(it.gseed)[idx], best, mark);
        if (hit == kGrazeMark) {
          best = glb(it.gseed)[idx];
          mark = MODE == 0 && !BVH && it.repair_run > 0;
        }
      }
    }
    thi = MODE == 2 ? widened(tmax)
                    : best == kMissKey ? kInf : widened(fkey_inv((uint32_t)(best >> 32)));
    sp = sb = 0;
    cur = 0u;  // interior node 0 (the root)
    pl = kDone;
  };
  // Evaluates the newest `cnt` (at most 64) candidates, one per lane; wavefront-uniform.
  auto run_chains = [&](uint32_t cnt) {
    const uint32_t e = qn - cnt + (uint32_t)lane;
    const bool have = (uint32_t)lane < cnt;
    bool failed = false;
    uint32_t ri = 0, job = 0;
    if (have) {
      ri = sQIdx[e];
      job = sQJob[e];
      const RhItem& it = item(job);
      const uint32_t ref = sQRef[e];
      const bool ok = chain(it, ri, ref);
      if constexpr (MODE == 2) {
        if (ok) glb(it.occ)[ri] = 1;
      } else if (direct) {
        if (ok) write_hit(it.r, it.v9, it.uv6, ri, (int32_t)ref, 0.f, it.out, false, true);
      } else {
        // stores of one wavefront to one address keep their order
        if (!ok) glb(it.keys)[ri] = kMissKey;
      }
      failed = !ok;
    }
    qn -= cnt;
    const uint64_t fb = __ballot(failed);
    if (failed) {
      const uint32_t p = kChainQ - 1u - nf - (uint32_t)__popcll(fb & lanes_below);
      sQIdx[p] = ri;
      sQJob[p] = (uint16_t)job;
    }
    nf += (uint32_t)__popcll(fb);
    __syncthreads();
  };
  for (;;) {
    // deal rays to the lanes without one: first those to trace again, then the queue's
    for (;;) {
      const uint64_t need = __ballot(!act);
      if (need == 0 || (more && nf == 0 && (uint32_t)__popcll(need) < kDealLanes)) break;
      const uint32_t rank = (uint32_t)__popcll(need & lanes_below);
      bool got = false;
      if (nf > 0) {
        const uint32_t take = min(nf, (uint32_t)__popcll(need));
        if (!act && rank < take) {
          idx = sQIdx[kChainQ - nf + rank];
          jk = sQJob[kChainQ - nf + rank];
          careful = true;
          got = true;
        }
        nf -= take;
        __syncthreads();
      } else {
        if (!more) break;
        // the lane's job, block, chunk of the block and slot in it
        uint32_t job = 0xffffffffu, blk = 0, part = 0, q = 0;
        if (spread != 0) {
          // the wavefront's only rays: `spread` of them in runs of at most 16, one run in each
          // of the launch's equal parts; consecutive wavefronts of an XCD take neighbouring runs
          more = false;
          const uint32_t run = min(spread, 16u);
          const uint32_t w = (blockIdx.x % (uint32_t)kClaimQueues) * (gridDim.x / kClaimQueues) +
                             blockIdx.x / (uint32_t)kClaimQueues;
          const uint32_t slot = ((uint32_t)lane / run * gridDim.x + w) * run + (uint32_t)lane % run;
          uint32_t c = slot / 64u;
          q = slot % 64u;
          if ((uint32_t)lane < spread && c < nchunks) {
            if (direct) {
              job = ONE ? 0u : find_chunk_item_lane(items, nitems, c);
              c -= item(job).chunk_base;
            } else {
              const uint2 v = rq[c];
              job = v.x;  // ~0u: a block-path block
              c = v.y;
            }
            if (job != 0xffffffffu) {
              const uint32_t nch = ((uint32_t)item(job).g.rb + 63u) / 64u;
              blk = c / nch;
              part = c - blk * nch;
            }
          }
        } else {
          if (cslot >= 64u) {
            uint32_t e = 0;
            if (lane == 0) e = claim_unit(ctr, nchunks, claim, 1);
            e = __builtin_amdgcn_readfirstlane(e);
            if (e >= nchunks) {
              more = false;
              break;
            }
            uint32_t c;
            if (direct) {
              cjob = ONE ? 0u : (uint32_t)find_chunk_item(items, nitems, e);
              c = e - item(cjob).chunk_base;
            } else {
              const uint2 w = rq[e];
              cjob = __builtin_amdgcn_readfirstlane(w.x);
              if (cjob == 0xffffffffu) continue;  // a block-path block
              c = __builtin_amdgcn_readfirstlane(w.y);
            }
            const uint32_t nch = ((uint32_t)item(cjob).g.rb + 63u) / 64u;
            cblk = c / nch;
            cpart = c - cblk * nch;
            cslot = 0;
          }
          q = cslot + rank;
          if (q < 64u) job = cjob;
          blk = cblk;
          part = cpart;
          cslot += min(64u - cslot, (uint32_t)__popcll(need));
        }
        if (!act && job != 0xffffffffu) {
          const RhItem& it = item(job);
          const RHGeom& g = it.g;
          const int gwt = g.gw[g.L - 1];
          const int J = (int)blk / gwt, K = (int)blk - J * gwt;
          int x = 0, y = 0, leaf = 0;
          if (slot_xy(g, K, J, (int)(part * 64u + q), x, y, leaf)) {
            idx = (uint32_t)y * (uint32_t)g.W + (uint32_t)x;
            jk = job;
            careful = false;
            got = it.ntri > 0 &&
                  (MODE == 0 || it.r.valid == nullptr || glb(it.r.valid)[idx] != 0);
            if (direct && !got) write_miss(it, idx);
            // occluded by the grazing pass
            if (MODE == 2 && got && it.gblock != nullptr && glb(it.gblock)[blk] == kGrazeHit)
              got = glb(it.occ)[idx] == 0;
          }
        }
      }
      if (got) {
        const RhItem& it = item(jk);
        const RaysDev& r = it.r;
        o = {glb(r.ox)[idx], glb(r.oy)[idx], glb(r.oz)[idx]};
        d = {glb(r.dx)[idx], glb(r.dy)[idx], glb(r.dz)[idx]};
        tmin = glb(r.tmin)[idx];
        tmax = glb(r.tmax)[idx];
        sr = slab_ray(F3{o.x, o.y, o.z}, F3{d.x, d.y, d.z}, it.sframe);
        tlo = tmin - fabsf(tmin) * kSlack;
        track_rep = MODE == 0 && !BVH && it.repair_run > 0;
        const bool again = careful;
        restart();
        careful = again;
        act = true;
      }
    }
    if (!__any(act)) {
      if (qn == 0) break;  // nothing to trace again either: the deal takes those first
      run_chains(min(qn, 64u));
      continue;
    }
    if (!more && nf == 0) {
      const uint64_t am = __ballot(act);
      if ((uint32_t)__popcll(am) <= kSplitLanes) {
        if (!split) {
          split = true;
          own = (uint32_t)lane;
          sRay[lane] = 1u | (mark ? kRayMark : 0u);
          if constexpr (MODE != 2) sBest[lane] = best;
          __syncthreads();
        }
        const bool gives = act && !careful && sp > sb;
        const uint64_t gm = __ballot(gives);
        const uint32_t n = min((uint32_t)__popcll(gm), (uint32_t)__popcll(~am));
        if (n > 0) {
          // the r-th giving lane and the r-th idle lane meet in entry 64 + r of the queue, which
          // holds less than 64 candidates here and nothing to trace again
          const uint32_t gr = (uint32_t)__popcll(gm & lanes_below);
          const uint32_t ir = (uint32_t)__popcll(~am & lanes_below);
          if (gives && gr < n) {
            sQIdx[64 + gr] = sStk[sb++][lane];
            sQRef[64 + gr] = (uint32_t)lane;
            atomicAdd(&sRay[own], 1u);
          }
          __syncthreads();
          const bool takes = !act && ir < n;
          const int from = takes ? (int)sQRef[64 + ir] : lane;
          auto copy = [&](auto& v) { v = __shfl(v, from); };
          copy(o.x); copy(o.y); copy(o.z);
          copy(d.x); copy(d.y); copy(d.z);
          copy(sr.ih.x); copy(sr.ih.y); copy(sr.ih.z);
          copy(sr.cn.x); copy(sr.cn.y); copy(sr.cn.z);
          copy(sr.cf.x); copy(sr.cf.y); copy(sr.cf.z);
          copy(tmin); copy(tmax); copy(tlo); copy(thi);
          copy(idx); copy(jk); copy(own);
          const bool tr = __shfl((int)track_rep, from) != 0;
          if constexpr (MODE != 2) {
            const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(best >> 32), from),
                           lo = (uint32_t)__shfl((int)(uint32_t)best, from);
            best = ((uint64_t)hi << 32) | lo;
          }
          if (takes) {
            act = true;
            careful = false;
            mark = false;
            track_rep = tr;
            sp = sb = 0;
            pl = kDone;
            cur = sQIdx[64 + ir];
            if (cur & kSearchLeafBit) {
              pl = cur;
              cur = kDone;
            }
          }
          __syncthreads();
        }
      }
    }
    const RhItem& it = item(jk);
    const auto snode = glb(it.snode);
    const auto tmts = glb(it.tmts);
    // node phase: a lane visits one 4-wide node a step, four 16-byte loads of one line, its
    // FP16 planes read by mixed-precision FMAs.  The walk is bound by the chain of dependent
    // node loads and by VALU issue at part-filled wavefronts; four children a node halve the
    // steps of the binary walk (FP32 boxes, 64 bytes a node): 1 M random segments against
    // 200,000 triangles 1,206 -> 1,089 us, room task to path depth 3, closest 855 -> 790 and
    // occlusion 2,516 -> 2,278 us, camera rays of twelve scenes 1,186 -> 1,049 us.
    for (;;) {
      if (act && cur != kDone && !(cur & kSearchLeafBit)) {
        const uint4 nx = ldu4(snode, 4 * (size_t)cur), ny = ldu4(snode, 4 * (size_t)cur + 1),
                    nz = ldu4(snode, 4 * (size_t)cur + 2), nm = ldu4(snode, 4 * (size_t)cur + 3);
        uint32_t key[4];
        node_keys(nx, ny, nz, nm, sr, tlo, thi, key);
        const uint32_t ni = nm.x >> 24;
        auto ref = [&](uint32_t k) {
          const uint32_t c = k & 3u;
          return (c < ni ? nm.y : nm.z) + c;
        };
        key_swap(key[0], key[1]);
        key_swap(key[2], key[3]);
        key_swap(key[0], key[2]);
        key_swap(key[1], key[3]);
        key_swap(key[1], key[2]);
        if (key[3] != kNoChild) sStk[sp++][lane] = ref(key[3]);
        if (key[2] != kNoChild) sStk[sp++][lane] = ref(key[2]);
        if (key[1] != kNoChild) sStk[sp++][lane] = ref(key[1]);
        cur = key[0] != kNoChild ? ref(key[0]) : pop();
        if (pl == kDone && cur != kDone && (cur & kSearchLeafBit)) {
          pl = cur;
          cur = pop();
        }
      }
      // walk on while more than walk64 / 64 of the lanes holding a ray have neither a postponed
      // leaf nor finished (fewer lanes idle behind the longest walk); the others go on from
      // their node in the next round (every round walks at least one step, so each lane
      // advances)
      const uint32_t searching = (uint32_t)__popcll(
          __ballot(act && pl == kDone && cur != kDone && !(cur & kSearchLeafBit)));
      if (64u * searching <= walk64 * (uint32_t)__popcll(__ballot(act))) break;
    }
    // leaf phase: the triangle each lane holds
    bool push = false;
    if (act && pl != kDone) {
      const uint32_t slot = pl & ~kSearchLeafBit;
      const float4 ta = ld4(tmts, 3 * (size_t)slot), tb = ld4(tmts, 3 * (size_t)slot + 1),
                   tc = ld4(tmts, 3 * (size_t)slot + 2);
      Tri T;
      T.v1 = {ta.x, ta.y, ta.z};
      T.e1 = {ta.w, tb.x, tb.y};
      T.e2 = {tb.z, tb.w, tc.x};
      T.v2 = T.v3 = T.v1;
      const uint32_t id = __float_as_uint(tc.y);
      const uint32_t bl = __float_as_uint(tc.z);  // ray-bvh: the triangle's reference BVH leaf
      // in no leaf; or not its leaf's first primitive (6DB / IA secondary rays)
      const bool ok = !BVH || (bl != 0xffffffffu &&
                               !(MODE == 1 && NODE != 2 && (bl & 0x80000000u)));
      const uint32_t ref = BVH && MODE == 2 ? bl & 0x7fffffffu : id;
      float t, b1, b2;
      if (ok && mt_strict(o, d, T, t, b1, b2)) {
        if constexpr (MODE == 2) {
          if (t > tmin && t < tmax) {  // intersectAllLeaves.cl:177-179
            if (!careful) {
              cand = ref;
              push = !split || !(atomicOr(&sRay[own], kRayMark) & kRayMark);
              act = push;  // false: another lane of the split ray has its candidate
            } else if (chain(it, idx, ref)) {
              glb(it.occ)[idx] = 1;
              act = false;
            }
          }
        } else {
          const bool main = t > tmin && t < kInf;
          const bool rp = track_rep && repair_kept(t, tmin) && repair_region(b1, b2);
          const uint64_t key = hit_key(t, (int32_t)id);
          const bool um = main && key < best;
          if ((um || (rp && !mark)) && (!careful || chain(it, idx, id))) {
            if (um) {
              best = key;
              thi = widened(t);
              if (split && !careful) atomicMin(&sBest[own], (unsigned long long)key);
            }
            if (rp) mark = true;
          }
        }
      }
      pl = kDone;
    }
    if (act && pl == kDone && cur != kDone && (cur & kSearchLeafBit)) {  // a second leaf waits
      pl = cur;
      cur = pop();
    }
    // rays that are done: a verified result is written; the others queue their candidate, if
    // they have one (a split ray's last lane for all of them)
    if (act && !push && cur == kDone && pl == kDone) {
      bool last = true;
      if (split && !careful) {
        if (MODE != 2 && mark) atomicOr(&sRay[own], kRayMark);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint32_t was = atomicAdd(&sRay[own], 0xffffffffu);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        last = (was & kRayLanes) == 1u && !(MODE == 2 && (was & kRayMark));
        if constexpr (MODE != 2) {
          best = lds_load(&sBest[own]);
          mark = (was & kRayMark) != 0u;
        }
      }
      const float tstar = best == kMissKey ? kInf : fkey_inv((uint32_t)(best >> 32));
      // whether the repair pass can change the ray (rh_finalize_kernel's rule; where t - EPS
      // rounds to t it is not asked which hit lies in the repair region)
      const bool repairs = MODE == 0 && track_rep &&
                           ((mark && !(tmin > tstar - kEps)) ||
                            (best != kMissKey && !(tstar > tstar - kEps)));
      if (!last) {
        act = false;
      } else if constexpr (MODE == 2) {
        if (direct) write_miss(it, idx);
        act = false;
      } else if (careful) {
        if (direct) {
          if (best == kMissKey) write_miss(it, idx);
          else write_hit(it.r, it.v9, it.uv6, idx, (int32_t)(uint32_t)best, tstar, it.out);
          if (repairs) replist[atomicAdd(&ctr[2], 1u)] = it.ray_base + idx;
        } else {
          if (best != kMissKey) glb(it.keys)[idx] = best;
          if (repairs) glb(it.repkeys)[idx] = fkey(mark ? tmin : tstar);
        }
        act = false;
      } else if (repairs) {
        restart();
      } else if (best == kMissKey) {
        if (direct) write_miss(it, idx);
        act = false;
      } else {
        push = true;
      }
    }
    const uint64_t pb = __ballot(push);
    if (pb != 0) {
      const uint32_t e = qn + (uint32_t)__popcll(pb & lanes_below);
      const bool room = e < kChainQ - nf;
      if (push) {
        if (room) {
          sQIdx[e] = idx;
          sQRef[e] = MODE == 2 ? cand : (uint32_t)best;
          sQJob[e] = (uint16_t)jk;
          if constexpr (MODE != 2) {
            if (!direct) glb(it.keys)[idx] = best;
          }
          act = false;
        } else {
          restart();
        }
      }
      qn = min(qn + (uint32_t)__popcll(pb), kChainQ - nf);
      __syncthreads();
      if (qn >= 64u) run_chains(64u);
    }
    // the other lanes' news of a split ray
    if (split && act && !careful) {
      if constexpr (MODE == 2) {
        if (lds_load(&sRay[own]) & kRayMark) act = false;
      } else {
        const uint64_t b = lds_load(&sBest[own]);
        if (b < best) {
          best = b;
          thi = widened(fkey_inv((uint32_t)(b >> 32)));
        }
      }
    }
  }
}

// Triangle staged in LDS as v1 and the two edges (the leaf test's operands).
__device__ __forceinline__ void stage_tri(float4 (*sT)[3], int slot, const Tri& T) {
  sT[slot][0] = make_float4(T.v1.x, T.v1.y, T.v1.z, T.e1.x);
  sT[slot][1] = make_float4(T.e1.y, T.e1.z, T.e2.x, T.e2.y);
  sT[slot][2] = make_float4(T.e2.z, 0.f, 0.f, 0.f);
}
__device__ __forceinline__ Tri staged_tri(const float4 (*sT)[3], int slot) {
  float4 a = sT[slot][0], b = sT[slot][1], c = sT[slot][2];
  Tri T;
  T.v1 = {a.x, a.y, a.z};
  T.e1 = {a.w, b.x, b.y};
  T.e2 = {b.z, b.w, c.x};
  T.v2 = T.v3 = T.v1;  // unused by the leaf test
  return T;
}

// ---------------------------------------------------------------------------------------
// Hit record of one ray from its reduction key; returns t (INFINITY on a miss).
__device__ __forceinline__ float finalize_ray(const RaysDev& r, const float* __restrict__ v9,
                                              const float* __restrict__ uv6, uint64_t key,
                                              size_t i, const HitOut& out,
                                              bool naive_rule = false) {
  if (key == kMissKey) {
    write_hit(r, v9, uv6, i, -1, 0.f, out);
    return __int_as_float(0x7f800000);
  }
  const float t = fkey_inv((uint32_t)(key >> 32));
  write_hit(r, v9, uv6, i, (int32_t)(uint32_t)key, t, out, naive_rule);
  return t;
}

// ---------------------------------------------------------------------------------------
// Naive brute force (naive.cl "TriRay" semantics, ray-parallel).
constexpr int kNaiveThreads = 512;
constexpr int kNaiveTris = 512;          // triangles staged at a time
constexpr int kNaiveShift = 6;           // 1 << kNaiveShift lanes test one triangle
constexpr int kNaiveRays = 2 << kNaiveShift;  // rays of a work-group: two to a lane

// A triangle as the naive kernel stages it.  With m = o x d the leaf test's numerators and
// determinant are linear in (d, m), so a ray is rejected by fused multiply-adds alone:
//   div = d.(e2 x e1), n1 = m.e2 - d.(e2 x v1), n2 = d.(e1 x v1) - m.e1.
// q[0] = e2 x e1 and the bound's factor (below), q[1] and q[2] = e2 and e2 x v1 + (e2 x e1) / 2,
// then e1 and e1 x v1; q[4] = v1.
struct NaiveTri {
  float4 q[5];
};
// |.|1 is the sum of magnitudes, u = 2^-24.  The rounding errors of n1 - div / 2 and |div| / 2 as
// the leaf test and as the filter compute them come to less than
// 20 u |d|1 (|e1|1 + |e2|1) (|o|1 + |v1|1 + |e1|1 + |e2|1), those of n2, n1 + n2 likewise to less
// than 28 u of it; the bound is 64 u.  Every norm counts as 2^-40 at least, which covers what
// underflow takes away (2^-150 times one of the factors), and where a factor exceeds 2^40, so
// that products could overflow, or is not a number, the bound is infinite: nothing is rejected.
constexpr float kNormMin = 0x1p-40f, kNormMax = 0x1p40f, kNaiveErr = 0x1p-18f;
__device__ __forceinline__ float norm1(V3 a) { return fabsf(a.x) + fabsf(a.y) + fabsf(a.z); }
__device__ __forceinline__ float norm_bound(float x) {
  return x <= kNormMax ? (x < kNormMin ? kNormMin : x) : __int_as_float(0x7f800000);
}

__device__ __forceinline__ void stage_naive(NaiveTri& s, const Tri& T, float omax) {
  const V3 n = cross(T.e2, T.e1), c1 = cross(T.e2, T.v1), c2 = cross(T.e1, T.v1);
  const float edges = norm1(T.e1) + norm1(T.e2), e = edges < kNormMin ? kNormMin : edges;
  const float f = norm_bound(e * (omax + norm1(T.v1) + e)) * kNaiveErr;
  s.q[0] = make_float4(n.x, n.y, n.z, f);
  s.q[1] = make_float4(T.e2.x, T.e2.y, T.e2.z, c1.x + 0.5f * n.x);
  s.q[2] = make_float4(c1.y + 0.5f * n.y, c1.z + 0.5f * n.z, T.e1.x, T.e1.y);
  s.q[3] = make_float4(T.e1.z, c2.x, c2.y, c2.z);
  s.q[4] = make_float4(T.v1.x, T.v1.y, T.v1.z, 0.f);
}
__device__ __forceinline__ float dot_fma(float x, float y, float z, V3 v, float c) {
  return __builtin_fmaf(x, v.x, __builtin_fmaf(y, v.y, __builtin_fmaf(z, v.z, c)));
}
// First part of the filter: false if b1 is certainly outside the leaf test's interval.
__device__ __forceinline__ bool naive_b1(const float4 (&q)[3], V3 d, V3 m, float dn, float half,
                                         float& div, float& err, float& x) {
  div = dot_fma(q[0].x, q[0].y, q[0].z, d, 0.f);
  x = dot_fma(q[1].x, q[1].y, q[1].z, m, -dot_fma(q[1].w, q[2].x, q[2].y, d, 0.f));
  err = dn * q[0].w;
  return !(fabsf(x) > __builtin_fmaf(half, fabsf(div), err));
}

// A work-group has the whole answer of its rays, two to a lane (a triangle's LDS reads serve two
// tests).  1 << shift lanes test one triangle; the parts of that many lanes share out the
// triangles, staged through LDS.  So a call is one launch, without keys in memory to clear,
// reduce by atomics and turn into hit records by launches of their own.
// Bound by vector issue: the leaf test alone takes 26 instructions to its first reject, the
// filter 12.  1,024 triangles, 128 x 128 rays: closest 24.5 -> 21 us and occlusion 27.6 -> 22 us
// (without the launches saved), 4,096 triangles, 250 x 200 rays: 392 -> 240 us for both.
template <int MODE>
__global__ __launch_bounds__(kNaiveThreads) void naive_kernel(RaysDev r,
                                                              const float* __restrict__ v9,
                                                              const float* __restrict__ uv6,
                                                              uint32_t ntri, int shift,
                                                              uint32_t chunk,
                                                              uint64_t* __restrict__ merge,
                                                              HitOut out, bool naive_rule,
                                                              uint8_t* __restrict__ occ_out) {
  constexpr bool P = MODE == 2;
  constexpr float half = naive_half<P>();
  __shared__ NaiveTri sT[kNaiveTris];
  __shared__ uint64_t sBest[kNaiveRays];  // closest: reduction key; occlusion: 0 when occluded
  __shared__ uint32_t sFar;               // largest |o|1 of the work-group's rays
  const int tid = threadIdx.x;
  const size_t n = (size_t)r.W * r.H;
  const int lanes = 1 << shift;
  const int slot = tid & (lanes - 1);
  const uint32_t part = (uint32_t)tid >> shift, parts = (uint32_t)kNaiveThreads >> shift;
  const size_t first = (size_t)blockIdx.x * (2 * lanes);
  if (tid < 2 * lanes) sBest[tid] = kMissKey;
  if (tid == 0) sFar = __float_as_uint(kNormMin);
  __syncthreads();
  V3 o[2], d[2], m[2];
  float tmin[2], tmax[2], dn[2];
  uint64_t best[2] = {kMissKey, kMissKey};
  bool live[2];
  for (int j = 0; j < 2; ++j) {
    const size_t i = first + slot + j * lanes;
    live[j] = i < n && (MODE == 0 || r.valid == nullptr || r.valid[i] != 0);
    o[j] = d[j] = {0.f, 0.f, 0.f};
    tmin[j] = tmax[j] = 0.f;
    if (live[j]) {
      o[j] = {r.ox[i], r.oy[i], r.oz[i]};
      d[j] = {r.dx[i], r.dy[i], r.dz[i]};
      tmin[j] = r.tmin[i];
      if (P) tmax[j] = r.tmax[i];
      // magnitudes order as their bit patterns do, NaN above all
      if (part == 0) atomicMax(&sFar, __float_as_uint(norm1(o[j])));
    }
    m[j] = cross(o[j], d[j]);
    dn[j] = norm_bound(norm1(d[j]));
  }
  const uint32_t tend = min(ntri, (blockIdx.y + 1) * chunk);
  for (uint32_t base = blockIdx.y * chunk; base < tend; base += kNaiveTris) {
    const uint32_t cnt = min(tend - base, (uint32_t)kNaiveTris);
    __syncthreads();
    const float omax = __uint_as_float(sFar);
    for (uint32_t k = tid; k < cnt; k += kNaiveThreads)
      stage_naive(sT[k], load_tri(v9, base + k), omax);
    __syncthreads();
    if (part >= cnt) continue;
    float4 q[3] = {sT[part].q[0], sT[part].q[1], sT[part].q[2]};
    for (uint32_t k = part; k < cnt; k += parts) {
      if (P && !__any(live[0] || live[1])) break;
      const uint32_t kn = k + parts < cnt ? k + parts : k;
      const float4 next[3] = {sT[kn].q[0], sT[kn].q[1], sT[kn].q[2]};
      for (int j = 0; j < 2; ++j) {
        float div, err, x;
        if (!naive_b1(q, d[j], m[j], dn[j], half, div, err, x) || !live[j]) continue;
        const float4 q3 = sT[k].q[3], q4 = sT[k].q[4];
        Tri T;
        T.v1 = T.v2 = T.v3 = {q4.x, q4.y, q4.z};
        T.e1 = {q[2].z, q[2].w, q3.x};
        T.e2 = {q[1].x, q[1].y, q[1].z};
        // b2 and b1 + b2, from x = n1 - div / 2; a determinant within the bound may have the
        // other sign or, without an inverse, make b1 NaN, after which no sum is rejected
        const float n2 = dot_fma(q3.y, q3.z, q3.w, d[j], -dot_fma(T.e1.x, T.e1.y, T.e1.z, m[j], 0.f));
        const float n12 = x + n2;
        const bool neg = div < 0.f;
        if (fabsf(div) > err &&
            ((neg ? -n2 : n2) < -__builtin_fmaf(half - 0.5f, fabsf(div), err) ||
             (neg ? -n12 : n12) > __builtin_fmaf(half, fabsf(div), err) + err))
          continue;
        float t;
        if (!mt_naive<P>(o[j], d[j], T, t) || t < tmin[j]) continue;
        if (P) {
          if (t > tmax[j]) continue;
          live[j] = false;
          best[j] = 0;
        } else {
          const uint64_t key = hit_key(t, (int32_t)(base + k));
          if (key < best[j]) best[j] = key;
        }
      }
      for (int c = 0; c < 3; ++c) q[c] = next[c];
    }
  }
  __syncthreads();
  for (int j = 0; j < 2; ++j)
    if (best[j] != kMissKey)
      atomicMin((unsigned long long*)&sBest[slot + j * lanes], (unsigned long long)best[j]);
  __syncthreads();
  const size_t i = first + tid;
  if (gridDim.y > 1) {  // naive_finish_kernel has the rest
    if (tid < 2 * lanes && sBest[tid] != kMissKey)
      atomicMin((unsigned long long*)&merge[i], (unsigned long long)sBest[tid]);
    return;
  }
  if (tid >= 2 * lanes || i >= n) return;
  if (P)
    occ_out[i] = sBest[tid] == 0 ? 1 : 0;
  else
    finalize_ray(r, v9, uv6, sBest[tid], i, out, naive_rule);
}

// Results of a naive launch whose triangles several work-groups shared out.
template <bool P>
__global__ __launch_bounds__(kThreads) void naive_finish_kernel(RaysDev r,
                                                                const float* __restrict__ v9,
                                                                const float* __restrict__ uv6,
                                                                const uint64_t* __restrict__ merge,
                                                                HitOut out, bool naive_rule,
                                                                uint8_t* __restrict__ occ_out) {
  const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= (size_t)r.W * r.H) return;
  if (P)
    occ_out[i] = merge[i] == 0 ? 1 : 0;
  else
    finalize_ray(r, v9, uv6, merge[i], i, out, naive_rule);
}

// Hit records of every job of a closest-hit group.  Rays whose nearest repair-region
// candidate lies at or below tHit - EPS are listed for the repair pass (only those can
// change, see rh_repair_kernel).
__global__ __launch_bounds__(256) void rh_finalize_kernel(const RhItem* __restrict__ items,
                                                          int nitems, uint32_t nrays,
                                                          uint32_t* __restrict__ ctr,
                                                          uint32_t* __restrict__ replist) {
  const uint32_t gi = blockIdx.x * kThreads + threadIdx.x;
  if (gi >= nrays) return;
  const RhItem& it = items[find_ray_item(items, nitems, gi)];
  const uint32_t i = gi - it.ray_base;
  const float tstar = finalize_ray(it.r, it.v9, it.uv6, it.keys[i], i, it.out);
  if (it.repkeys) {
    const uint32_t rk = it.repkeys[i];
    if (rk != kNoKey32 && !(fkey_inv(rk) > tstar - kEps)) replist[atomicAdd(&ctr[2], 1u)] = gi;
  }
}

// Exact sequential repair pass (yetAnotherIntersection6DB.cl with repairRun passes, in
// increasing triangle id order) for the rays whose outcome it can change: the nearest
// repair-region candidate lies at or below tHit - EPS (hits at exactly tmin, or ties at t
// large enough that t - EPS rounds to t).  One work-group per flagged ray.
template <int NODE>
__global__ __launch_bounds__(256) void rh_repair_kernel(const RhItem* __restrict__ items,
                                                        int nitems,
                                                        const uint32_t* __restrict__ ctr,
                                                        const uint32_t* __restrict__ replist) {
  __shared__ Node sChain[kMaxLevels];
  __shared__ int sWc[kThreads / 64];
  __shared__ float sEt[kThreads];
  __shared__ uint32_t sEi[kThreads];
  __shared__ float sTH;
  __shared__ int sIdx;
  const int tid = threadIdx.x, lane = __lane_id(), wave = tid >> 6;
  const uint32_t count = ctr[2];
  for (uint32_t w = blockIdx.x; w < count; w += gridDim.x) {
    const uint32_t gi = __builtin_amdgcn_readfirstlane(replist[w]);
    const RhItem& it = items[find_ray_item(items, nitems, gi)];
    const RHGeom& g = it.g;
    const RaysDev& r = it.r;
    const float* __restrict__ v9 = it.v9;
    const uint32_t ntri = it.ntri;
    const size_t i = gi - it.ray_base;
    const int x = (int)(i % (size_t)g.W), y = (int)(i / (size_t)g.W);
    if (tid < g.L) {
      const int l = tid;
      const int gk = x / (g.cx << l), gj = y / (g.cy << l);
      const float4* p = it.nodes + 4 * ((size_t)g.off[l] + (size_t)gj * g.gw[l] + gk);
      float4 a = ld4(p, 0), b = ld4(p, 1), c = ld4(p, 2), d = ld4(p, 3);
      sChain[l].dmin = {a.x, a.y, a.z};
      sChain[l].dmax = {b.x, b.y, b.z};
      sChain[l].omin = {c.x, c.y, c.z};
      sChain[l].omax = {d.x, d.y, d.z};
    }
    if (tid == 0) {
      sTH = it.out.t[i];
      sIdx = it.out.id[i];
    }
    __syncthreads();
    const V3 o = {r.ox[i], r.oy[i], r.oz[i]};
    const V3 d = {r.dx[i], r.dy[i], r.dz[i]};
    const float tmin = r.tmin[i];
    for (int run = 0; run < it.repair_run; ++run) {
      for (uint32_t base = 0; base < ntri; base += kThreads) {
        const uint32_t ti = base + tid;
        bool have = false;
        float t = 0.f;
        if (ti < ntri) {
          const Tri T = load_tri(v9, ti);
          bool pass = true;
          if (NODE != 0) {
            const V3 bmin = vmin(vmin(T.v1, T.v2), T.v3), bmax = vmax(vmax(T.v1, T.v2), T.v3);
            for (int l = g.L - 1; l >= 0 && pass; --l)
              pass = NODE == 1 ? cull_ia(sChain[l], bmin, bmax) : cull_5db(sChain[l], bmin, bmax);
          } else {
            for (int l = g.L - 1; l >= 0 && pass; --l) pass = cull_tri(sChain[l], T);
          }
          float b1, b2;
          if (pass && mt_strict(o, d, T, t, b1, b2) && repair_region(b1, b2) && t >= tmin)
            have = true;
        }
        const uint64_t bal = __ballot(have);
        const int prefix = __popcll(bal & ((1ull << lane) - 1ull));
        if (lane == 0) sWc[wave] = __popcll(bal);
        __syncthreads();
        int woff = 0, total = 0;
        for (int k = 0; k < kThreads / 64; ++k) {
          if (k < wave) woff += sWc[k];
          total += sWc[k];
        }
        if (have) {
          sEt[woff + prefix] = t;
          sEi[woff + prefix] = ti;
        }
        __syncthreads();
        if (tid == 0) {
          for (int e = 0; e < total; ++e) {
            if (sEt[e] > sTH - kEps || (int)sEi[e] == sIdx) continue;
            sTH = sEt[e];
            sIdx = (int)sEi[e];
          }
        }
        __syncthreads();
      }
    }
    if (tid == 0) write_hit(r, v9, it.uv6, i, sIdx, sTH, it.out);
    __syncthreads();
  }
}

// Shadow rays toward a point light (light.h:79-84, point.cpp:42-49).
// When `count` is given, the number of valid shadow rays is added to it.
__global__ __launch_bounds__(256) void shadow_kernel(RaysDev pr, const int32_t* __restrict__ id,
                                                     const float* __restrict__ tt, float lx,
                                                     float ly, float lz, float* ox, float* oy,
                                                     float* oz, float* dx, float* dy, float* dz,
                                                     float* tmin, float* tmax, uint8_t* valid,
                                                     uint32_t* count) {
  const size_t n = (size_t)pr.W * pr.H;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (count) {
    const uint64_t bal = __ballot(i < n && id[i] >= 0);
    if (__lane_id() == 0 && bal) atomicAdd(count, (uint32_t)__popcll(bal));
  }
  if (i >= n) return;
  if (id[i] < 0) {
    ox[i] = oy[i] = oz[i] = 0.f;
    dx[i] = dy[i] = dz[i] = 0.f;
    tmin[i] = tmax[i] = 0.f;
    valid[i] = 0;
    return;
  }
  const float t = tt[i];
  const float px = pr.ox[i] + pr.dx[i] * t;
  const float py = pr.oy[i] + pr.dy[i] * t;
  const float pz = pr.oz[i] + pr.dz[i] * t;
  const float vx = lx - px, vy = ly - py, vz = lz - pz;
  const float dist = sqrtf((vx * vx + vy * vy) + vz * vz);
  const float inv = 1.f / dist;
  ox[i] = px;
  oy[i] = py;
  oz[i] = pz;
  dx[i] = vx * inv;
  dy[i] = vy * inv;
  dz[i] = vz * inv;
  tmin[i] = 1e-3f * t;
  tmax[i] = dist * (1.f - 0.f);
  valid[i] = 1;
}

// Pinhole camera rays of a render request: image (W*spp) x H, the spp samples of a pixel
// adjacent in x (the reference sampler's order); pixel centres for spp == 1, otherwise a
// counter-based hash of (seed, x, y, sample) gives the jitter.  The FP32 operation order is
// that of the workloads' numpy camera, so spp == 1 images are identical to it.
__device__ __forceinline__ uint32_t mix32(uint32_t h) {
  h ^= h >> 16;
  h *= 0x7feb352du;
  h ^= h >> 15;
  h *= 0x846ca68bu;
  h ^= h >> 16;
  return h;
}
__global__ __launch_bounds__(256) void camera_kernel(int W, int H, int spp, float cx, float cy,
                                                     float cz, float tan_half, float aspect,
                                                     uint32_t seed, float* ox, float* oy,
                                                     float* oz, float* dx, float* dy, float* dz,
                                                     float* tmin, float* tmax) {
  const size_t n = (size_t)W * spp * H;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int row = W * spp;
  const int y = (int)(i / (size_t)row), c = (int)(i % (size_t)row);
  const int x = c / spp, k = c % spp;
  float jx = 0.5f, jy = 0.5f;
  if (spp > 1) {
    const uint32_t h = mix32(seed ^ mix32((uint32_t)x * 0x9e3779b9u ^ mix32((uint32_t)y ^
                                                                          ((uint32_t)k << 20))));
    jx = (float)(h >> 8) * (1.0f / 16777216.0f);
    jy = (float)(mix32(h) >> 8) * (1.0f / 16777216.0f);
  }
  const float px = ((((float)x + jx) / (float)W) * 2.0f - 1.0f) * tan_half * aspect;
  const float py = (1.0f - (((float)y + jy) / (float)H) * 2.0f) * tan_half;
  const float pz = 1.0f;
  const float l = sqrtf((px * px + py * py) + pz * pz);
  const float inv = 1.0f / l;
  ox[i] = cx;
  oy[i] = cy;
  oz[i] = cz;
  dx[i] = px * inv;
  dy[i] = py * inv;
  dz[i] = pz * inv;
  tmin[i] = 0.f;
  tmax[i] = __int_as_float(0x7f800000);
}

// Path-tracing bounce rays from closest hits: origin p = o + d*t, a cosine-weighted direction
// about the geometric normal of the hit triangle turned toward the incoming ray, tmin =
// 1e-3*t (pbrt's rayEpsilon), tmax = INFINITY; random numbers hashed from (seed, ray, depth)
// so the rays do not depend on the launch order.
__global__ __launch_bounds__(256) void bounce_kernel(RaysDev in, const float* __restrict__ v9,
                                                     const int32_t* __restrict__ id,
                                                     const float* __restrict__ tt, uint32_t seed,
                                                     int depth, float* ox, float* oy, float* oz,
                                                     float* dx, float* dy, float* dz,
                                                     float* tmin, float* tmax, uint8_t* valid) {
  const size_t n = (size_t)in.W * in.H;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t tri = id[i];
  if (tri < 0 || (in.valid != nullptr && in.valid[i] == 0)) {
    ox[i] = oy[i] = oz[i] = 0.f;
    dx[i] = dy[i] = dz[i] = 0.f;
    tmin[i] = tmax[i] = 0.f;
    valid[i] = 0;
    return;
  }
  const float t = tt[i];
  const V3 d = {in.dx[i], in.dy[i], in.dz[i]};
  const V3 p = {in.ox[i] + d.x * t, in.oy[i] + d.y * t, in.oz[i] + d.z * t};
  const Tri T = load_tri(v9, (uint32_t)tri);
  V3 nn = normalize(cross(T.e1, T.e2));
  if (dot(nn, d) > 0.f) nn = {-nn.x, -nn.y, -nn.z};
  const uint32_t h = mix32(seed ^ mix32((uint32_t)i * 0x9e3779b9u ^ mix32((uint32_t)depth)));
  const float u1 = (float)(h >> 8) * (1.0f / 16777216.0f);
  const float u2 = (float)(mix32(h) >> 8) * (1.0f / 16777216.0f);
  const float r = sqrtf(u1), phi = 6.28318530717958647692f * u2;
  const float lx = r * cosf(phi), ly = r * sinf(phi), lz = sqrtf(fmaxf(0.f, 1.f - u1));
  // orthonormal basis about nn (Duff et al. 2017)
  const float sgn = nn.z >= 0.f ? 1.f : -1.f;
  const float a = -1.f / (sgn + nn.z);
  const float b = nn.x * nn.y * a;
  const V3 t1 = {1.f + sgn * nn.x * nn.x * a, sgn * b, -sgn * nn.x};
  const V3 t2 = {b, sgn + nn.y * nn.y * a, -nn.y};
  const V3 w = {t1.x * lx + t2.x * ly + nn.x * lz, t1.y * lx + t2.y * ly + nn.y * lz,
                t1.z * lx + t2.z * ly + nn.z * lz};
  ox[i] = p.x;
  oy[i] = p.y;
  oz[i] = p.z;
  dx[i] = w.x;
  dy[i] = w.y;
  dz[i] = w.z;
  tmin[i] = 1e-3f * t;
  tmax[i] = __int_as_float(0x7f800000);
  valid[i] = 1;
}

template <class T>
__global__ void fill_kernel(T* p, T v, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

inline dim3 grid1(size_t n) { return dim3((unsigned)((n + kThreads - 1) / kThreads)); }

// Work-groups of a persistent kernel that are resident at once on the current device: CUs x
// work-groups per CU (limited by registers and LDS) for `threads`-wide work-groups, at most
// `cap`.  A larger grid only adds work-groups that start when the queue is nearly drained.
// The count is kept per (device, kernel) once known (2048 until then).
template <class F>
unsigned resident_grid(F kernel, uint32_t cap, int threads = kThreads) {
  static std::mutex mu;
  static std::map<std::pair<int, const void*>, unsigned> known;
  int dev = 0;
  unsigned n = 0;
  const bool have_dev = hipGetDevice(&dev) == hipSuccess;
  const std::pair<int, const void*> key{dev, reinterpret_cast<const void*>(kernel)};
  if (have_dev) {
    std::lock_guard<std::mutex> lk(mu);
    auto f = known.find(key);
    if (f != known.end()) n = f->second;
  }
  if (n == 0) {
    int cus = 0, per_cu = 0;
    if (have_dev &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) ==
            hipSuccess &&
        cus > 0 && per_cu > 0) {
      n = (unsigned)cus * (unsigned)per_cu;
      std::lock_guard<std::mutex> lk(mu);
      known[key] = n;
    } else {
      n = 2048;
    }
  }
  return std::max(1u, std::min(n, std::max(cap, 1u)));
}

// RT_PARAM_WALK_* as 64ths of the lanes holding a ray: 1/2^v, none for 7.  The built-in 3/8 was the
// fastest or within 2% of it on every workload measured (1 M segments: 7/8 of the lanes 856 us,
// 3/4 775, 1/2 688, 1/4 688, 1/8 770; with the lanes of a wavefront better filled, camera rays of
// twelve scenes 555 us at 1/2, 538 at 3/8, 527 at 1/4).
constexpr uint32_t kWalk64[8] = {24, 32, 16, 8, 4, 2, 1, 0};

// Launch sequence of one rayhierarchy group with the mode and node type fixed.
template <int MODE, int NODE>
hipError_t rh_group_dispatch(const RhGroup& G, hipStream_t s, const RhEvents& ev) {
  auto record = [&](hipEvent_t e) { return e ? hipEventRecord(e, s) : hipSuccess; };
  hipError_t e = record(ev.first);
  if (e != hipSuccess) return e;
  const bool direct = G.ray_clusters == 0;  // every block ray by ray, results written there
  if (!direct)
    hipLaunchKernelGGL((rh_init_kernel<MODE>), grid1(std::max<uint32_t>(G.nrays, kClaimQueues)),
                       dim3(kThreads), 0, s, G.items, G.nitems, G.nrays, G.ctr);
  uint32_t* const clear = direct ? G.ctr : nullptr;
  auto build = [&](auto group, auto single) {
    if (G.single)
      hipLaunchKernelGGL(single, dim3(G.nblocks), dim3(kThreads), 0, s, *G.single,
                         const_cast<RhItem*>(G.items), clear);
    else
      hipLaunchKernelGGL(group, dim3(G.nblocks), dim3(kThreads), 0, s, G.items, G.nitems, clear);
  };
  if (G.one_ray)
    build(rh_group_build_kernel<MODE != 0, NODE == 2, true>,
          rh_single_build_kernel<MODE != 0, NODE == 2, true>);
  else
    build(rh_group_build_kernel<MODE != 0, NODE == 2, false>,
          rh_single_build_kernel<MODE != 0, NODE == 2, false>);
  e = hipGetLastError();
  if (e == hipSuccess && direct) e = record(ev.trace);
  if (e != hipSuccess) return e;
  if (direct) {
    if (G.graze) {
      const dim3 grid(std::min<uint32_t>(G.nblocks, kGrazeGrid));
      auto launch = [&](auto kernel, int waves) {
        if (G.graze == 2) {  // few blocks
          hipLaunchKernelGGL(kernel, dim3(G.nblocks * kGrazeSlices), dim3(64 * waves), 0, s, G.items,
                             G.nitems, G.nblocks, G.ctr, G.heavy, (uint32_t)kGrazeSlices, false);
          return;
        }
        hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), 0, s, G.items, G.nitems, G.nblocks,
                           G.ctr, G.heavy, 1u, false);
        hipLaunchKernelGGL(kernel, dim3(kGrazeSecond), dim3(64 * waves), 0, s, G.items, G.nitems,
                           G.nblocks, G.ctr, G.heavy, (uint32_t)kGrazeSlices, true);
      };
      if (G.bvh) launch(rh_graze_kernel<MODE, NODE, true, 4>, 4);
      else launch(rh_graze_kernel<MODE, NODE, false, 4>, 4);
    }
  } else if (G.bvh)
    hipLaunchKernelGGL((rh_cluster_kernel<MODE, NODE, true>), dim3(G.nblocks), dim3(kThreads), 0,
                       s, G.items, G.nitems, G.ustage, G.bunits, G.rq, G.ctr, G.per_unit,
                       G.ray_clusters);
  else
    hipLaunchKernelGGL((rh_cluster_kernel<MODE, NODE, false>), dim3(G.nblocks), dim3(kThreads),
                       0, s, G.items, G.nitems, G.ustage, G.bunits, G.rq, G.ctr, G.per_unit,
                       G.ray_clusters);
  if (G.ray_clusters > 1) {  // 1 sends every block with work per-ray: no unit
    hipLaunchKernelGGL(rh_unit_scan_kernel, dim3((G.nblocks + kScanThreads - 1) / kScanThreads),
                       dim3(kScanThreads), 0, s, G.bunits, G.nblocks);
    hipLaunchKernelGGL(rh_unit_pack_kernel, dim3((G.nblocks + kPackThreads / 64 - 1) /
                                                 (kPackThreads / 64)),
                       dim3(kPackThreads), 0, s, G.bunits, G.nblocks, G.ustage, G.units, G.ctr);
  }
  e = hipGetLastError();
  if (e == hipSuccess && !direct) e = record(ev.trace);
  if (e == hipSuccess) e = record(ev.ready);
  if (e != hipSuccess) return e;
  auto launch = [&](auto kernel) {
    const dim3 grid(G.grid > 0 ? (unsigned)G.grid : resident_grid(kernel, G.max_units));
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, s, G.items, G.units, G.ctr);
  };
  if (direct) {
  } else if (G.bvh && G.big)
    launch(bvh_unit_kernel<MODE, NODE, 1024, 4>);
  else if (G.bvh)
    launch(bvh_unit_kernel<MODE, NODE, 256, 3>);
  else if (G.big)
    launch(rh_unit_kernel<MODE, NODE, 1024, 4>);
  else
    launch(rh_unit_kernel<MODE, NODE, 256, 3>);
  e = hipGetLastError();
  if (e == hipSuccess) e = record(ev.ray);
  if (e != hipSuccess) return e;
  auto launch_rays = [&](auto kernel) {
    unsigned spread = 0;
    const unsigned slots = resident_grid(kernel, 0x7fffffffu, 64);
    const dim3 grid = [&]() {
      if (G.ray_grid > 0) return std::max(1u, std::min((unsigned)G.ray_grid, G.max_chunks));
      if (G.max_chunks > slots) return slots;
      const unsigned rays = G.max_chunks * 64u;
      spread = (rays + slots - 1) / slots;
      spread = spread > 16 ? (spread + 15) / 16 * 16 : spread > 8 ? 16 : spread > 4 ? 8 : 4;
      return ((rays + spread - 1) / spread + kClaimQueues - 1) / kClaimQueues * kClaimQueues;
    }();
    hipLaunchKernelGGL(kernel, grid, dim3(64), 0, s, G.items, G.nitems,
                       direct ? nullptr : G.rq, G.ctr, G.replist, G.max_chunks, spread,
                       kWalk64[std::min(std::max(G.walk, 0), 7)]);
  };
  if (G.nitems == 1) {
    if (G.bvh) launch_rays(ray_path_kernel<MODE, NODE, true, true>);
    else launch_rays(ray_path_kernel<MODE, NODE, false, true>);
  } else {
    if (G.bvh) launch_rays(ray_path_kernel<MODE, NODE, true, false>);
    else launch_rays(ray_path_kernel<MODE, NODE, false, false>);
  }
  e = hipGetLastError();
  if (e == hipSuccess) e = record(ev.ray_end);
  if (e != hipSuccess) return e;
  if (MODE != 2) {
    if (!direct)
      hipLaunchKernelGGL(rh_finalize_kernel, grid1(G.nrays), dim3(kThreads), 0, s, G.items,
                         G.nitems, G.nrays, G.ctr, G.replist);
    if (MODE == 0 && G.replist && !G.bvh)
      hipLaunchKernelGGL((rh_repair_kernel<NODE>), dim3(64), dim3(kThreads), 0, s, G.items,
                         G.nitems, G.ctr, G.replist);
  }
  e = hipGetLastError();
  return e == hipSuccess ? record(ev.last) : e;
}

// See launch_graze_records.
__global__ __launch_bounds__(256) void graze_records_kernel(
    const float* __restrict__ v9, const uint32_t* __restrict__ order,
    const uint32_t* __restrict__ tleaf, uint32_t n, SearchFrame frame,
    GrazeNormal* __restrict__ normal, GrazeTri* __restrict__ out, float4* __restrict__ test) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const uint32_t id = order[i];
  float p[9];
  for (int k = 0; k < 9; ++k) p[k] = v9[9 * (size_t)id + k];
  out[i] = graze_record(p, id, frame);
  normal[i] = graze_normal(out[i], frame);
  const Tri T = load_tri(v9, id);
  test[3 * (size_t)i] = make_float4(T.v1.x, T.v1.y, T.v1.z, T.e1.x);
  test[3 * (size_t)i + 1] = make_float4(T.e1.y, T.e1.z, T.e2.x, T.e2.y);
  test[3 * (size_t)i + 2] = make_float4(T.e2.z, __uint_as_float(id),
                                        __uint_as_float(tleaf ? tleaf[id] : 0u),
                                        graze_near_slope(out[i], normal[i]));
}
__global__ __launch_bounds__(256) void graze_clusters_kernel(const GrazeTri* __restrict__ rec,
                                                             const uint32_t* __restrict__ first,
                                                             uint32_t n, uint32_t nclusters,
                                                             GrazeCluster* __restrict__ out) {
  const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= nclusters) return;
  const uint32_t a = first ? first[c] : c * (uint32_t)kCluster;
  const uint32_t z = first ? first[c + 1] : min(n, a + (uint32_t)kCluster);
  out[c] = graze_cluster(rec + a, z - a);
}

// See launch_set_tleaf.
__global__ __launch_bounds__(256) void set_tleaf_kernel(float4* __restrict__ tmts,
                                                        const uint32_t* __restrict__ tleaf,
                                                        uint32_t ntri) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= ntri) return;
  float4& r = tmts[3 * (size_t)i + 2];
  r.z = __uint_as_float(tleaf[__float_as_uint(r.y)]);
}

// Scratch of the allocation-free trace (rt_trace_closest_noalloc): one array per device, held
// until the process ends.  Its device address is looked up in this file, once per device.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratch];

}  // namespace

// Device address of `scratch` on each device, looked up by noalloc_setup.
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices] = {};

int noalloc_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return 1;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return 0;
  int cur = -1;
  if (hipGetDevice(&cur) != hipSuccess || cur != device) return 1;  // the device must be current
  void* p = nullptr;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return 1;
  g_scratch_ptr[device] = p;
  return 0;
}

void* noalloc_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return g_scratch_ptr[device];
}

hipError_t launch_graze_records(const float* v9, const uint32_t* order, const uint32_t* tleaf,
                                uint32_t n, const uint32_t* first, uint32_t nclusters,
                                const SearchFrame& frame, GrazeNormal* normal, GrazeTri* out,
                                float4* test, GrazeCluster* cout, hipStream_t s) {
  if (n)
    hipLaunchKernelGGL(graze_records_kernel, grid1(n), dim3(kThreads), 0, s, v9, order, tleaf, n,
                       frame, normal, out, test);
  if (nclusters)
    hipLaunchKernelGGL(graze_clusters_kernel, grid1(nclusters), dim3(kThreads), 0, s, out, first,
                       n, nclusters, cout);
  return hipGetLastError();
}

hipError_t launch_set_tleaf(float4* tmts, const uint32_t* tleaf, uint32_t ntri, hipStream_t s) {
  if (!ntri) return hipSuccess;
  hipLaunchKernelGGL(set_tleaf_kernel, grid1(ntri), dim3(kThreads), 0, s, tmts, tleaf, ntri);
  return hipGetLastError();
}

int rh_geometry(int W, int H, int cx, int cy, int height, RHGeom* g) {
  if (W <= 0 || H <= 0 || cx <= 0 || cy <= 0 || height <= 0) return 1;
  if (cx > (1 << 24) || cy > (1 << 24)) return 3;
  int gw = (int)(((int64_t)W + cx - 1) / cx), gh = (int)(((int64_t)H + cy - 1) / cy);
  g->W = W;
  g->H = H;
  g->cx = cx;
  g->cy = cy;
  g->gw[0] = gw;
  g->gh[0] = gh;
  int L = 1;
  // The level count is the reference's: it halves with floor and stops after a level whose
  // floor width or height is odd (rayhierarchy.cpp:412-442).  The grids themselves halve with
  // ceil, so a parent also covers the last child column (row) that the reference's floor
  // leaves out where it halves an odd dimension.
  int fw = gw, fh = gh;
  for (int i = 1; i < height; ++i) {
    if (L >= kMaxLevels) return 2;
    gw = (gw + 1) / 2;
    gh = (gh + 1) / 2;
    fw /= 2;
    fh /= 2;
    g->gw[L] = gw;
    g->gh[L] = gh;
    ++L;
    // a zero floor dimension leaves the reference no top-level node (it traces nothing):
    // stop there too
    if ((fw & 1) || (fh & 1) || fw == 0 || fh == 0) break;
  }
  g->L = L;
  int off = 0;
  for (int l = 0; l < L; ++l) {
    g->off[l] = off;
    off += g->gw[l] * g->gh[l];
  }
  g->nnodes = off;
  g->nlx = 1 << (L - 1);
  if ((int64_t)cx * g->nlx * cy * g->nlx > kMaxRaysPerBlock) return 3;
  g->bw = cx * g->nlx;
  g->bh = cy * g->nlx;
  g->rb = g->bw * g->bh;
  g->g = cx * cy;
  g->nsub = ((1 << (2 * L)) - 1) / 3;
  g->ntop = g->gw[L - 1] * g->gh[L - 1];
  return 0;
}

hipError_t launch_fill_u8(uint8_t* p, uint8_t v, size_t n, hipStream_t s) {
  if (!n) return hipSuccess;
  hipLaunchKernelGGL(fill_kernel<uint8_t>, grid1(n), dim3(kThreads), 0, s, p, v, n);
  return hipGetLastError();
}

hipError_t launch_rh_group(const RhGroup& G, hipStream_t s, const RhEvents& ev) {
  if (G.nitems <= 0 || G.nrays == 0) return hipSuccess;
#define RT_CALL(M, N) rh_group_dispatch<M, N>(G, s, ev)
  if (G.node == 1) {
    if (G.mode == 0) return RT_CALL(0, 1);
    if (G.mode == 1) return RT_CALL(1, 1);
    return RT_CALL(2, 1);
  }
  if (G.node == 2) {
    if (G.mode == 0) return RT_CALL(0, 2);
    if (G.mode == 1) return RT_CALL(1, 2);
    return RT_CALL(2, 2);
  }
  if (G.mode == 0) return RT_CALL(0, 0);
  if (G.mode == 1) return RT_CALL(1, 0);
  return RT_CALL(2, 0);
#undef RT_CALL
}

// How a naive launch shares out rays and triangles.
struct NaiveShape {
  int shift = kNaiveShift;          // rays to a work-group: 2 << shift
  uint32_t groups = 1, parts = 1;   // work-groups over the rays, over the triangles
  uint32_t chunk = 0;               // triangles to a part
};
static NaiveShape naive_shape(size_t n, uint32_t ntri) {
  NaiveShape g;
  const auto groups = [&] { return (uint32_t)(((n - 1) >> (g.shift + 1)) + 1); };
  // Rays to a work-group: as many as leave 1,024 work-groups, four to a CU (three are resident
  // at once), and 8 at least.  4,096 triangles, 250 x 200 rays, both kernels: 512 work-groups
  // 266 us, 1,024 240, 2,048 254, 4,096 335 (every work-group stages all triangles); 128 x 128
  // rays equal.  With 128 rays always, 33 x 40 rays would leave 245 CUs idle.
  while (g.shift > 2 && groups() < kNaiveGroups) --g.shift;
  // Fewer than that, and enough triangles to pay for two launches more and the keys: as many
  // rays to a work-group again as leave 1,024 with the triangles shared out, since a triangle
  // is staged once for all of them.  Whole calls, shared by one work-group -> by several: 64
  // rays, 4,500 triangles 24 -> 27 us, 6,000 28 -> 27, 20,000 76 -> 27, 200,000 767 -> 27;
  // 1,024 rays, 20,000 triangles 80 -> 30, 200,000 724 -> 142 (with 8 rays each 224); 8,000
  // rays, 6,000 triangles 60 -> 50, 200,000 1,548 -> 1,032 (8 rays each 1,358).  The last to
  // arrive writing the results in the same launch took a fence a work-group, 300 us in all.
  uint32_t parts = 1;
  if (groups() < kNaiveGroups && ntri >= kNaiveSplit) {
    const uint32_t most = ntri / kNaiveTris;
    g.shift = kNaiveShift;
    while (g.shift > 2 && (size_t)groups() * most < kNaiveGroups) --g.shift;
    parts = std::min(most, (kNaiveGroups + groups() - 1) / groups());
  }
  while (g.shift > 0 && n <= ((size_t)1 << g.shift)) --g.shift;  // one group
  g.groups = groups();
  g.chunk = std::max((ntri + parts - 1) / parts, 1u);
  g.parts = std::max((ntri + g.chunk - 1) / g.chunk, 1u);
  return g;
}

hipError_t launch_naive_trace(const RaysDev& r, int mode, const float* v9, const float* uv6,
                              uint32_t ntri, bool naive_rule, uint64_t* merge, HitOut out,
                              uint8_t* occ, hipStream_t s) {
  const size_t n = (size_t)r.W * r.H;
  const NaiveShape g = naive_shape(n, ntri);
  if (g.parts > 1)
    hipLaunchKernelGGL(fill_kernel<uint64_t>, grid1(n), dim3(kThreads), 0, s, merge,
                       (uint64_t)kMissKey, n);
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(g.groups, g.parts), dim3(kNaiveThreads), 0, s, r, v9, uv6,
                       ntri, g.shift, g.chunk, merge, out, naive_rule, occ);
  };
  if (mode == 0) run(naive_kernel<0>);
  else if (mode == 1) run(naive_kernel<1>);
  else run(naive_kernel<2>);
  if (g.parts > 1) {
    auto finish = mode == 2 ? naive_finish_kernel<true> : naive_finish_kernel<false>;
    hipLaunchKernelGGL(finish, grid1(n), dim3(kThreads), 0, s, r, v9, uv6, merge, out, naive_rule,
                       occ);
  }
  return hipGetLastError();
}

hipError_t launch_camera_rays(int W, int H, int spp, const float origin[3], float tan_half,
                              float aspect, uint32_t seed, float* ox, float* oy, float* oz,
                              float* dx, float* dy, float* dz, float* tmin, float* tmax,
                              hipStream_t s) {
  const size_t n = (size_t)W * spp * H;
  hipLaunchKernelGGL(camera_kernel, grid1(n), dim3(kThreads), 0, s, W, H, spp, origin[0],
                     origin[1], origin[2], tan_half, aspect, seed, ox, oy, oz, dx, dy, dz, tmin,
                     tmax);
  return hipGetLastError();
}

hipError_t launch_bounce_rays(const RaysDev& in, const float* v9, const int32_t* id,
                              const float* t, uint32_t seed, int depth, float* ox, float* oy,
                              float* oz, float* dx, float* dy, float* dz, float* tmin,
                              float* tmax, uint8_t* valid, hipStream_t s) {
  const size_t n = (size_t)in.W * in.H;
  hipLaunchKernelGGL(bounce_kernel, grid1(n), dim3(kThreads), 0, s, in, v9, id, t, seed, depth,
                     ox, oy, oz, dx, dy, dz, tmin, tmax, valid);
  return hipGetLastError();
}

hipError_t launch_shadow_rays(const RaysDev& pr, const int32_t* id, const float* t, float lx,
                              float ly, float lz, float* ox, float* oy, float* oz, float* dx,
                              float* dy, float* dz, float* tmin, float* tmax, uint8_t* valid,
                              hipStream_t s, uint32_t* count) {
  const size_t n = (size_t)pr.W * pr.H;
  hipLaunchKernelGGL(shadow_kernel, grid1(n), dim3(kThreads), 0, s, pr, id, t, lx, ly, lz, ox,
                     oy, oz, dx, dy, dz, tmin, tmax, valid, count);
  return hipGetLastError();
}

}  // namespace rti
