// rt_search_bvh.cpp -- the search BVH of the per-ray path.
//
// Incoherent ray groups (random shadow rays, diffuse bounces) have direction boxes that cover
// most of the sphere, so the reference's cull chain keeps nearly every (leaf, triangle) pair
// of such a group and enumerating the candidate set costs a leaf test per pair.  The per-ray
// path finds the same answer from the other side: every candidate that can change a ray
// passes the strict leaf test, so each ray walks a BVH over the triangles, runs the strict
// leaf test on the triangles of the leaves it reaches, and evaluates the reference's exact
// cull chain only for triangles that pass it.  The BVH only has to be conservative: a box
// test may pass for a box the ray misses, never the other way round.
//
// A binary tree is built first and collapsed to four children per node.
//
// Binary tree: a binned SAH build over the triangles' bounding boxes, down to one triangle per
// leaf: 16 bins on each axis with a centroid extent, split cost nL * area(L) + nR * area(R) (the
// first minimum over the axes x, y, z in turn and the planes in order), stable partitions.  A
// range whose centroids coincide on every axis, or whose SAH split would take the tree past
// kSearchDepth interior levels, is split at the median by (centroid, id) on the axis of largest
// centroid extent.  Binning every axis in place of the widest one alone made the per-ray kernels
// about 4% faster on a batch of 64 cluster scenes.  Every box is the FP32 min/max of its
// triangles' vertices grown outward by pad = 2^-11 * max(1, largest vertex coordinate
// magnitude), more for thin triangles, which covers the rounding of the strict leaf test's hit
// point and of the slab test unless the ray grazes the triangle's plane (rt_search.h).
//
// Collapse: a wide node starts from a binary node's two children and replaces its interior child
// of largest area by that child's two children until it has four.  A ray loads about half as
// many nodes as in the binary tree (counted on the CPU: cluster scene of 200,000 triangles,
// camera rays 112.6 -> 57.1, random segments 58.8 -> 29.0; room, diffuse bounces 121.2 -> 58.4),
// and a walk is a chain of dependent loads.  An expansion is only made while the walk's stack
// stays within its entries: with k siblings left behind, every interior child must have at most
// (budget - k) binary levels below it, which any binary tree of no more levels than entries
// meets by keeping two children per node.
//
// Node planes are FP16 in units of the frame above the node's cell of a 256^3 grid over the
// scene, rounded outward: a relative step of 2^-11 of the node's own size plus one cell, i.e.
// at most 2^-19 of the scene for small nodes, so the boxes keep nearly the quality of FP32 ones
// in a 64-byte node (8-bit planes: 2% more nodes visited), and the kernel's mixed-precision FMA
// reads FP16 operands without a conversion instruction.  Vertices that are not finite never
// pass the strict leaf test; they are left out of the frame and the padding, and boxes reaching
// beyond the frame are cut to it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "rt_internal.h"

namespace rti {
namespace {

constexpr int kBins = 16;

struct SBox {
  float lo[3], hi[3];
  void clear() {
    for (int k = 0; k < 3; ++k) {
      lo[k] = INFINITY;
      hi[k] = -INFINITY;
    }
  }
  void grow(const SBox& b) {
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], b.lo[k]);
      hi[k] = std::max(hi[k], b.hi[k]);
    }
  }
  float area() const {
    const float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
    return 2.f * ((dx * dy + dy * dz) + dz * dx);
  }
};

struct Prim {
  SBox box;
  float c[3];  // centre of the box
};

// Interior levels a balanced (median split) tree needs over n triangles.
int levels_needed(uint32_t n) {
  int l = 0;
  while (n > 1) {
    n = (n + 1) / 2;
    ++l;
  }
  return l;
}

// Interior node of the binary tree: its children's boxes (padded) and references (bit 31: the
// leaf of that search position) and its interior levels.
struct BNode {
  SBox box[2];
  uint32_t ref[2];
  int levels;
};

class SearchBuilder {
 public:
  SearchBuilder(const std::vector<Prim>& prims, std::vector<uint32_t>& order,
                std::vector<BNode>& out, float pad)
      : P_(prims), idx_(order), out_(out), pad_(pad) {}

  // Reference of the subtree over search positions [a, b) whose parent sits at interior depth
  // `depth` (the root node is depth 1); its box (unpadded) goes to `box`.
  uint32_t build(uint32_t a, uint32_t b, int depth, SBox& box) {
    const uint32_t n = b - a;
    if (n == 1) return leaf(a, box);
    float clo[3] = {INFINITY, INFINITY, INFINITY}, chi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = a; i < b; ++i)
      for (int k = 0; k < 3; ++k) {
        clo[k] = std::min(clo[k], P_[idx_[i]].c[k]);
        chi[k] = std::max(chi[k], P_[idx_[i]].c[k]);
      }
    int ax = 0;  // widest centroid extent: the axis of a median split
    for (int k = 1; k < 3; ++k)
      if (chi[k] - clo[k] > chi[ax] - clo[ax]) ax = k;
    // the cheapest binned split over the three axes (the first minimum, axes in order)
    int best_ax = -1, best = -1;
    if (n == 2) {
      // every plane between the two costs the same: the first axis that tells them apart
      for (int axis = 2; axis >= 0; --axis)
        if (chi[axis] > clo[axis]) best_ax = axis;
      best = best_ax < 0 ? -1 : 0;
    } else {
      sah_split(a, b, clo, chi, best_ax, best);
    }
    bool median = best < 0;
    uint32_t m = 0;
    if (!median) {
      const float scale = (float)kBins / (chi[best_ax] - clo[best_ax]);
      const float lo = clo[best_ax];
      const int axis = best_ax, split = best;
      // stable: the left ones move down in place, the right ones through a buffer
      uint32_t* base = idx_.data();
      uint32_t* mid = base + a;
      tmp_.clear();
      for (uint32_t i = a; i < b; ++i) {
        const uint32_t t = base[i];
        if (bin(P_[t].c[axis], lo, scale) <= split) *mid++ = t;
        else tmp_.push_back(t);
      }
      std::copy(tmp_.begin(), tmp_.end(), mid);
      m = (uint32_t)(mid - base);
      if (m == a || m == b || depth + levels_needed(m - a) > kSearchDepth ||
          depth + levels_needed(b - m) > kSearchDepth)
        median = true;
    }
    if (median) {
      std::stable_sort(idx_.begin() + a, idx_.begin() + b, [&](uint32_t s0, uint32_t s1) {
        return P_[s0].c[ax] < P_[s1].c[ax] || (P_[s0].c[ax] == P_[s1].c[ax] && s0 < s1);
      });
      m = a + n / 2;
    }
    const uint32_t node = (uint32_t)out_.size();
    out_.emplace_back();
    SBox b0, b1;
    const uint32_t r0 = build(a, m, depth + 1, b0);
    const uint32_t r1 = build(m, b, depth + 1, b1);
    BNode& o = out_[node];
    o.box[0] = b0;
    o.box[1] = b1;
    for (int c = 0; c < 2; ++c)
      for (int k = 0; k < 3; ++k) {
        o.box[c].lo[k] -= pad_;
        o.box[c].hi[k] += pad_;
      }
    o.ref[0] = r0;
    o.ref[1] = r1;
    o.levels = 1 + std::max(levels(r0), levels(r1));
    box = b0;
    box.grow(b1);
    return node;
  }
  int levels(uint32_t ref) const { return ref & kSearchLeafBit ? 0 : out_[ref].levels; }

 private:
  static int bin(float c, float lo, float scale) {
    const float f = (c - lo) * scale;
    return f >= (float)(kBins - 1) ? kBins - 1 : f > 0.f ? (int)f : 0;  // NaN: 0
  }

  void sah_split(uint32_t a, uint32_t b, const float* clo, const float* chi, int& best_ax,
                 int& best) const {
    SBox bb[3][kBins];
    uint32_t cnt[3][kBins] = {};
    float scale[3];
    for (int axis = 0; axis < 3; ++axis) {
      const float ext = chi[axis] - clo[axis];
      scale[axis] = ext > 0.f ? (float)kBins / ext : 0.f;
      for (int k = 0; k < kBins; ++k) bb[axis][k].clear();
    }
    for (uint32_t i = a; i < b; ++i) {
      const Prim& p = P_[idx_[i]];
      for (int axis = 0; axis < 3; ++axis) {
        const int k = bin(p.c[axis], clo[axis], scale[axis]);
        bb[axis][k].grow(p.box);
        ++cnt[axis][k];
      }
    }
    float best_cost = INFINITY;
    for (int axis = 0; axis < 3; ++axis) {
      if (!(chi[axis] - clo[axis] > 0.f)) continue;
      float rarea[kBins];
      uint32_t rcnt[kBins];
      SBox acc;
      acc.clear();
      uint32_t c = 0;
      for (int k = kBins - 1; k > 0; --k) {
        if (cnt[axis][k]) {
          c += cnt[axis][k];
          acc.grow(bb[axis][k]);
          rarea[k] = acc.area();
        } else {
          rarea[k] = k < kBins - 1 ? rarea[k + 1] : 0.f;
        }
        rcnt[k] = c;
      }
      acc.clear();
      c = 0;
      for (int k = 0; k < kBins - 1; ++k) {
        if (!cnt[axis][k]) continue;  // the same split as the plane before: not cheaper
        c += cnt[axis][k];
        acc.grow(bb[axis][k]);
        if (rcnt[k + 1] == 0) break;
        const float cost = (float)c * acc.area() + (float)rcnt[k + 1] * rarea[k + 1];
        if (cost < best_cost) {
          best_cost = cost;
          best = k;
          best_ax = axis;
        }
      }
    }
  }

  uint32_t leaf(uint32_t a, SBox& box) const {
    box = P_[idx_[a]].box;
    return kSearchLeafBit | a;
  }

  const std::vector<Prim>& P_;
  std::vector<uint32_t>& idx_;
  std::vector<BNode>& out_;
  std::vector<uint32_t> tmp_;
  float pad_;
};

// FP16 bits of the nearest value at or below (up = false) or at or above (up = true) x, for
// 0 <= x < 65504.
uint32_t half_toward(double x, bool up) {
  if (!(x > 0.0)) return 0;
  uint64_t bits;
  std::memcpy(&bits, &x, 8);
  const int e = (int)(bits >> 52) - 1023;
  const uint64_t m = (bits & ((1ull << 52) - 1)) | (1ull << 52);
  // units of the last place: 2^(e - 10), at least 2^-24 (subnormals)
  const int drop = 42 + std::max(0, -14 - e);
  if (drop > 53) return up ? 1u : 0u;
  uint32_t q = (uint32_t)(m >> drop);
  if (up && (m & ((1ull << drop) - 1))) ++q;  // may carry into the exponent, as it should
  return e < -14 ? q : ((uint32_t)(e + 15) << 10) + q - 1024u;
}

// Collapses the binary tree into wide nodes; see the head of the file.
class Collapser {
 public:
  Collapser(const std::vector<BNode>& bin, const std::vector<uint32_t>& bin_order,
            const SearchFrame& frame, std::vector<uint4>& out, std::vector<uint32_t>& order)
      : B_(bin), bin_order_(bin_order), f_(frame), out_(out), order_(order) {}

  struct Child {
    SBox box;
    uint32_t ref;
  };
  void node(uint32_t at, Child* ch, int n, int budget) {
    while (n < 4) {
      int pick = -1;
      float area = -1.f;
      for (int i = 0; i < n; ++i) {
        if (ch[i].ref & kSearchLeafBit) continue;
        // the expansion leaves n siblings beside any child
        bool fits = true;
        for (int j = 0; j < n; ++j)
          if (j != i && levels(ch[j].ref) > budget - n) fits = false;
        if (levels(ch[i].ref) - 1 > budget - n) fits = false;
        const float s = ch[i].box.area();
        if (fits && !(s <= area)) {  // NaN areas too
          area = s;
          pick = i;
        }
      }
      if (pick < 0) break;
      const BNode& b = B_[ch[pick].ref];
      ch[pick] = Child{b.box[0], b.ref[0]};
      ch[n++] = Child{b.box[1], b.ref[1]};
    }
    std::stable_partition(ch, ch + n, [](const Child& c) { return !(c.ref & kSearchLeafBit); });
    int ni = 0;
    while (ni < n && !(ch[ni].ref & kSearchLeafBit)) ++ni;
    const uint32_t first = (uint32_t)(out_.size() / 4), tri = (uint32_t)order_.size();
    out_.resize(out_.size() + 4 * (size_t)ni);
    for (int i = ni; i < n; ++i) order_.push_back(bin_order_[ch[i].ref & ~kSearchLeafBit]);
    write(at, ch, n, ni, first, tri);
    for (int i = 0; i < ni; ++i) {
      const BNode& b = B_[ch[i].ref];
      Child c[4] = {Child{b.box[0], b.ref[0]}, Child{b.box[1], b.ref[1]}, {}, {}};
      node(first + (uint32_t)i, c, 2, budget - (n - 1));
    }
  }

  // Root over a single triangle.
  void single(const SBox& box) {
    Child c[4] = {Child{box, kSearchLeafBit}, {}, {}, {}};
    order_.push_back(bin_order_[0]);
    write(0, c, 1, 0, 0, 0);
  }

 private:
  int levels(uint32_t ref) const { return ref & kSearchLeafBit ? 0 : B_[ref].levels; }

  void write(uint32_t at, const Child* ch, int n, int ni, uint32_t first, uint32_t tri) {
    uint4* p = &out_[4 * (size_t)at];
    const double inv = 1.0 / (double)f_.unit;  // a power of two
    uint32_t cells = 0;
    for (int k = 0; k < 3; ++k) {
      // planes in frame units; a box is cut to the frame (non-finite ends included)
      double lo[4], hi[4], cell = 255.0;
      for (int i = 0; i < n; ++i) {
        lo[i] = ((double)ch[i].box.lo[k] - (double)f_.base[k]) * inv;
        hi[i] = ((double)ch[i].box.hi[k] - (double)f_.base[k]) * inv;
        if (!(lo[i] > 0.0)) lo[i] = 0.0;
        if (!(hi[i] < 256.0)) hi[i] = 256.0;
        cell = std::min(cell, std::floor(lo[i]));
      }
      cells |= (uint32_t)cell << (8 * k);
      uint32_t h[8];
      for (int i = 0; i < 4; ++i) {
        h[i] = i < n ? half_toward(lo[i] - cell, false) : 0x7bffu;
        h[4 + i] = i < n ? half_toward(hi[i] - cell, true) : 0xfbffu;
      }
      p[k] = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
    }
    p[3] = make_uint4(cells | (uint32_t)ni << 24, first, (kSearchLeafBit | tri) - (uint32_t)ni,
                      (uint32_t)n);
  }

  const std::vector<BNode>& B_;
  const std::vector<uint32_t>& bin_order_;
  const SearchFrame& f_;
  std::vector<uint4>& out_;
  std::vector<uint32_t>& order_;
};

}  // namespace

void build_search_bvh(const float* v9, uint32_t ntri, std::vector<uint4>& nodes,
                      std::vector<uint32_t>& order, SearchFrame& frame) {
  nodes.clear();
  order.clear();
  frame = SearchFrame{};
  frame.unit = 1.f;
  if (ntri == 0) return;
  std::vector<uint32_t> bin_order(ntri);
  for (uint32_t i = 0; i < ntri; ++i) bin_order[i] = i;
  float big = 1.f;
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (uint32_t i = 0; i < ntri; ++i) {
    const float* p = v9 + 9 * (size_t)i;
    for (int q = 0; q < 9; ++q) {
      if (!std::isfinite(p[q])) continue;
      big = std::max(big, std::fabs(p[q]));
      lo[q % 3] = std::min(lo[q % 3], (double)p[q]);
      hi[q % 3] = std::max(hi[q % 3], (double)p[q]);
    }
  }
  const float pad = std::ldexp(big, -11);
  frame.pad = pad;
  frame.huge = big > kGrazeHuge;
  double half2 = 0.0;
  for (int k = 0; k < 3; ++k) {
    if (!(lo[k] <= hi[k])) lo[k] = hi[k] = 0.0;
    frame.center[k] = (float)(0.5 * (lo[k] + hi[k]));
    const double h = std::max(hi[k] - frame.center[k], frame.center[k] - lo[k]);
    half2 += h * h;
  }
  std::vector<Prim> prims(ntri);
  float widest = pad;
  double edge2 = 0.0;
  for (uint32_t i = 0; i < ntri; ++i) {
    const float* p = v9 + 9 * (size_t)i;
    const float kappa = graze_record(p, i, frame).kappa;
    const float wide = pad * (pad_grow(kappa) - 1.f);  // what nodes add to `pad` for this one
    widest = std::max(widest, pad + wide);
    double s1 = 0.0, s2 = 0.0;
    for (int k = 0; k < 3; ++k) {
      prims[i].box.lo[k] = std::min(std::min(p[k], p[3 + k]), p[6 + k]) - wide;
      prims[i].box.hi[k] = std::max(std::max(p[k], p[3 + k]), p[6 + k]) + wide;
      prims[i].c[k] = (prims[i].box.lo[k] + prims[i].box.hi[k]) * 0.5f;
      s1 += ((double)p[3 + k] - p[k]) * ((double)p[3 + k] - p[k]);
      s2 += ((double)p[6 + k] - p[k]) * ((double)p[6 + k] - p[k]);
    }
    if (std::isfinite(s1)) edge2 = std::max(edge2, s1);
    if (std::isfinite(s2)) edge2 = std::max(edge2, s2);
  }
  frame.reach = (float)((std::sqrt(half2) + std::sqrt(edge2)) * (1.0 + 1e-6));
  // 255 units of a power of two span the padded scene from `base` on every axis
  double ext = 0.0;
  for (int k = 0; k < 3; ++k) {
    frame.base[k] = (float)(lo[k] - 2.0 * widest);
    ext = std::max(ext, hi[k] - lo[k] + 4.0 * widest);
  }
  int e;
  std::frexp(ext / 255.0, &e);
  frame.unit = std::ldexp(1.f, e);
  nodes.reserve(2 * (size_t)ntri);
  order.reserve(ntri);
  nodes.resize(4);
  std::vector<BNode> bin;
  bin.reserve(ntri);
  SearchBuilder b(prims, bin_order, bin, pad);
  Collapser w(bin, bin_order, frame, nodes, order);
  SBox box;
  if (ntri == 1) {
    box = prims[0].box;
    for (int k = 0; k < 3; ++k) {
      box.lo[k] -= pad;
      box.hi[k] += pad;
    }
    w.single(box);
    return;
  }
  b.build(0, ntri, 1, box);
  Collapser::Child c[4] = {Collapser::Child{bin[0].box[0], bin[0].ref[0]},
                           Collapser::Child{bin[0].box[1], bin[0].ref[1]}, {}, {}};
  w.node(0, c, 2, kSearchStack);
}

}  // namespace rti
