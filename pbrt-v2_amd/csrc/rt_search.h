// rt_search.h -- the geometry of the per-ray path's search tree, for its builder, the kernels and
// host code that walks the same tree: rays against its nodes, and which rays and triangles the
// tree cannot answer for.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace rti {

#define RT_HD __host__ __device__ __forceinline__

struct F3 {
  float x, y, z;
};

// Frame of a search tree: node planes (grid cell c of an axis starts at base + c * unit) and what
// bounds the rounding errors of leaf tests against its triangles.
struct SearchFrame {
  float base[3];
  float unit;
  float center[3];  // of the scene's vertices
  float reach;      // distance of the farthest vertex from the centre, plus the longest edge
  float pad;        // growth of the boxes of well-conditioned triangles
  int huge;         // coordinates beyond kGrazeHuge: no bound holds
};

constexpr float kSlack = 0x1p-16f;     // relative slack of the slab-test parameters
constexpr float kOffSlack = 0x1p-20f;  // the same of a ray's plane offsets

// ---------------------------------------------------------------------------------------
// Which strict hits the tree finds.
//
// A hit of the strict leaf test is found when its ray meets the triangle's padded box at the
// computed parameter.  With v1, e1, e2 the test's operands, R = |o - v1|, n = e1 x e2 and
// u = 2^-24, the roundings of the determinant d . n come to at most 6 u |d||e1||e2|, those of the
// numerators of b1, b2 and t to 7 u R |d||e2|, 7 u R |d||e1| and 7 u R |e1||e2|.  While |d . n|
// is well above its error, the exact ray meets the exact plane within
//   (14 R + 6 (|e1| + |e2|)) u |d||e1||e2| / |d . n|
// of the triangle, and the computed parameter lies within (13 R + 6 |e|) of the same of that
// point: together below 27 u rho kappa / sin(angle), where rho bounds R plus the longer edge's
// length, angle is the one between the ray and the triangle's plane and kappa = |e1||e2| / |n| >=
// 1 (1 / sine of the triangle's angle at v1).  It stays within 9/10 of the pad, the rest being
// left to the slab test's own roundings, if
//   sin(angle) >= A = 30 u kappa rho / pad.
// A ray that grazes the plane at less may pass the test by its roundings alone, anywhere along
// that plane, and no pad covers it.  But the ray then runs close to the plane all the way: with
// |n1|, |n2| <= |d . n| + errors, the origin is within
//   rho (A + 13 u) lambda / cos(angle)
// of it, lambda = 1 / sin(half the angle between the lines of e1 and e2), which is 1 / (the larger
// sine of the angles that the ray's projection makes with them) or more.
//
// Rays at an angle of A / kGrazeNear or more are still near the triangle, within kGrazeNear pads
// (with 13 R + 6 |e| grown by what the point itself is off, as long as that is below rho / 2);
// only below it the distance bound, with A / kGrazeNear, is all there is.
//
// Triangles with kappa above kGrazeKappa have a pad up to kGrazeGrow times wider, so that thin
// ones do not make every ray a grazing one; and rays from so far that their errors outgrow the
// pad widen all boxes for themselves (ray_pad), which keeps 30 u rho / pad below 0.03.
constexpr float kGrazeKappa = 4.f, kGrazeGrow = 64.f;
constexpr float kGrazeNear = 16.f;
constexpr float kGrazeErr = 33.f * 0x1p-24f;  // 30 u and a tenth for the roundings of the bounds
constexpr float kFarPad = 6e-5f;              // pad for a unit of rho
constexpr float kGrazeHuge = 1e10f;           // beyond it products of three lengths may overflow
// Directions shorter or longer, and products of edges below, may lose digits to underflow.
constexpr float kGrazeDirMin = 1e-6f, kGrazeDirMax = 1e6f, kGrazeEdges = 1e-24f;

// A triangle as the grazing pass sees it.
struct GrazeTri {
  float n[3];   // unit normal
  float h;      // n . (v1 - frame centre)
  float kappa;  // negative: no ray passes its test; infinite: every ray may graze it
  float lambda;
  uint32_t id;  // original triangle
  float reach;  // |v1 - frame centre| plus the longer edge
  float v[3];   // v1 - frame centre
  float edge;   // the longer edge
};

RT_HD float pad_grow(float kappa) {  // the pad of a triangle, in frame pads
  const float g = kappa * (1.f / kGrazeKappa);
  return g > 1.f ? (g < kGrazeGrow ? g : kGrazeGrow) : 1.f;
}

// p: v1, v2, v3.  kappa is rounded up.
RT_HD GrazeTri graze_record(const float* p, uint32_t id, const SearchFrame& f) {
  GrazeTri g{};
  g.id = id;
  g.kappa = -1.f;
  double e1[3], e2[3], l1 = 0, l2 = 0, c = 0, bad = 0;
  for (int k = 0; k < 3; ++k) {
    const float a = p[3 + k] - p[k], b = p[6 + k] - p[k];  // the test's operands
    e1[k] = a;
    e2[k] = b;
    l1 += e1[k] * e1[k];
    l2 += e2[k] * e2[k];
    c += e1[k] * e2[k];
    bad += 0.0 * (double)p[k] + 0.0 * (double)a + 0.0 * (double)b;  // NaN if not finite
  }
  if (!(bad == 0.0)) return g;
  if (!(l1 > 0.0) || !(l2 > 0.0)) return g;  // the determinant is exactly zero
  const double nx = e1[1] * e2[2] - e1[2] * e2[1], ny = e1[2] * e2[0] - e1[0] * e2[2],
               nz = e1[0] * e2[1] - e1[1] * e2[0];
  const double len = sqrt(nx * nx + ny * ny + nz * nz), edges = sqrt(l1) * sqrt(l2);
  const double vx = (double)p[0] - f.center[0], vy = (double)p[1] - f.center[1],
               vz = (double)p[2] - f.center[2];
  g.v[0] = (float)vx;
  g.v[1] = (float)vy;
  g.v[2] = (float)vz;
  g.edge = (float)(sqrt(fmax(l1, l2)) * (1.0 + 1e-6));
  g.reach = (float)((sqrt(vx * vx + vy * vy + vz * vz) + g.edge) * (1.0 + 1e-6));
  g.kappa = INFINITY;
  if (f.huge || !(len > 0.0) || !(edges >= (double)kGrazeEdges)) return g;
  const double kappa = edges / len;
  if (!(kappa < 1e6)) return g;
  g.kappa = (float)(kappa * (1.0 + 1e-6));
  const double cosine = fmin(fabs(c) / edges, 1.0);
  g.lambda = (float)(2.0 * sqrt(0.5 * (1.0 + cosine)) * kappa * (1.0 + 1e-6));
  g.n[0] = (float)(nx / len);
  g.n[1] = (float)(ny / len);
  g.n[2] = (float)(nz / len);
  g.h = (float)((nx * vx + ny * vy + nz * vz) / len);
  return g;
}

// The width by which a ray whose origin is `dist` away from the frame's centre grows every box.
RT_HD float ray_pad(float dist, const SearchFrame& f) {
  const float w = kFarPad * (dist + f.reach) - f.pad;
  return w > 0.f ? w : 0.f;
}

// Square root and reciprocal to one unit in the last place or better; every use has a margin.
RT_HD float near_sqrt(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_sqrtf(x);
#else
  return sqrtf(x);
#endif
}
RT_HD float near_rcp(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.f / x;
#endif
}

// Boxes of a set of rays: origins and far points (any point of the ray) relative to the frame's
// centre, and directions; and what the pass's bounds need of them.
struct GrazeRays {
  F3 oc, oh, qc, qh, dc, dh;  // centres and half widths
  float dist, far, dir;       // bounds of |origin|, of |far point - origin|, of |d|
  float extra;                // the least ray_pad
  bool all;                   // no bound holds: every triangle may be grazed
};
RT_HD void graze_axis(float lo, float hi, float ref, float& c, float& h) {
  const float a = lo - ref, b = hi - ref;
  c = 0.5f * (a + b);
  h = 0.5f * (b - a) + 0x1p-21f * (fabsf(a) + fabsf(b));  // and the roundings of a, b and c
}
// dmin: the smallest of the rays' largest direction components.
RT_HD GrazeRays graze_rays(const float* olo, const float* ohi, const float* qlo, const float* qhi,
                           const float* dlo, const float* dhi, float dmin, const SearchFrame& f) {
  GrazeRays r;
  graze_axis(olo[0], ohi[0], f.center[0], r.oc.x, r.oh.x);
  graze_axis(olo[1], ohi[1], f.center[1], r.oc.y, r.oh.y);
  graze_axis(olo[2], ohi[2], f.center[2], r.oc.z, r.oh.z);
  graze_axis(qlo[0], qhi[0], f.center[0], r.qc.x, r.qh.x);
  graze_axis(qlo[1], qhi[1], f.center[1], r.qc.y, r.qh.y);
  graze_axis(qlo[2], qhi[2], f.center[2], r.qc.z, r.qh.z);
  graze_axis(dlo[0], dhi[0], 0.f, r.dc.x, r.dh.x);
  graze_axis(dlo[1], dhi[1], 0.f, r.dc.y, r.dh.y);
  graze_axis(dlo[2], dhi[2], 0.f, r.dc.z, r.dh.z);
  const F3 o = {fabsf(r.oc.x) + r.oh.x, fabsf(r.oc.y) + r.oh.y, fabsf(r.oc.z) + r.oh.z};
  const F3 d = {fabsf(r.dc.x) + r.dh.x, fabsf(r.dc.y) + r.dh.y, fabsf(r.dc.z) + r.dh.z};
  const F3 q = {fabsf(r.qc.x - r.oc.x) + r.qh.x + r.oh.x, fabsf(r.qc.y - r.oc.y) + r.qh.y + r.oh.y,
                fabsf(r.qc.z - r.oc.z) + r.qh.z + r.oh.z};
  const F3 n = {fmaxf(fabsf(r.oc.x) - r.oh.x, 0.f), fmaxf(fabsf(r.oc.y) - r.oh.y, 0.f),
                fmaxf(fabsf(r.oc.z) - r.oh.z, 0.f)};
  r.dist = near_sqrt(o.x * o.x + o.y * o.y + o.z * o.z) * (1.f + 0x1p-20f);
  r.dir = near_sqrt(d.x * d.x + d.y * d.y + d.z * d.z) * (1.f + 0x1p-20f);
  r.far = near_sqrt(q.x * q.x + q.y * q.y + q.z * q.z) * (1.f + 0x1p-20f);
  r.extra = ray_pad(near_sqrt(n.x * n.x + n.y * n.y + n.z * n.z) * (1.f - 0x1p-20f), f);
  r.all = !(dmin >= kGrazeDirMin && r.dir <= kGrazeDirMax && r.dist <= kGrazeHuge);
  return r;
}
// Whether some line through the box c +- h in the set's directions may come within w of v on every
// axis: the parameters at which the axis of the steadiest direction gets there, then the other two
// axes at those.
RT_HD bool comes_near(const GrazeRays& r, const F3& c, const F3& h, const float* v, float w) {
  const F3 ad = {fabsf(r.dc.x) - r.dh.x, fabsf(r.dc.y) - r.dh.y, fabsf(r.dc.z) - r.dh.z};
  const bool ux = ad.x >= ad.y && ad.x >= ad.z, uy = !ux && ad.y >= ad.z;
  // main axis first
  const float a = ux ? ad.x : uy ? ad.y : ad.z;
  if (!(a > 0.f)) return true;
  const float s0 = ux ? v[0] - c.x : uy ? v[1] - c.y : v[2] - c.z;
  const float h0 = (ux ? h.x : uy ? h.y : h.z) + w;
  const float dc0 = ux ? r.dc.x : uy ? r.dc.y : r.dc.z, dh0 = ux ? r.dh.x : uy ? r.dh.y : r.dh.z;
  const float s1 = ux ? v[1] - c.y : v[0] - c.x, s2 = ux || uy ? v[2] - c.z : v[1] - c.y;
  const float o1 = ux ? h.y : h.x, o2 = ux || uy ? h.z : h.y;
  const float dc1 = ux ? r.dc.y : r.dc.x, dh1 = ux ? r.dh.y : r.dh.x;
  const float dc2 = ux || uy ? r.dc.z : r.dc.y, dh2 = ux || uy ? r.dh.z : r.dh.y;
  // parameters t0 +- th at which the main axis is reached, then the offset there
  const float far = (fabsf(s0) + h0) * near_rcp(a) * (1.f + 0x1p-20f), inv = near_rcp(dc0);
  const float t0 = s0 * inv;
  const float th = (far * dh0 + h0) * fabsf(inv) * (1.f + 0x1p-18f) + far * 0x1p-18f;
  const float e = 0x1p-18f * (fabsf(s0) + fabsf(s1) + fabsf(s2) + w + far * r.dir);
  const float m1 = fabsf(s1 - t0 * dc1), m2 = fabsf(s2 - t0 * dc2);
  if (m1 > o1 + w + e + far * dh1 + th * fabsf(dc1)) return false;
  return !(m2 > o2 + w + e + far * dh2 + th * fabsf(dc2));
}
// Whether any of the rays may graze the triangle, in two parts that both have to pass: by angle
// and distance of its plane, and by its place.  Every comparison lets a NaN through.  low: the
// first part passes even at A / kGrazeNear.
RT_HD bool grazes_plane(const GrazeRays& r, const float* n, float h, float kappa, float lambda,
                        float reach, const SearchFrame& f, bool& low) {
  low = true;
  if (kappa < 0.f) return false;
  const float rho = r.dist + reach;
  const float P = pad_grow(kappa) * f.pad + r.extra, kw = kappa * (kGrazeErr * rho);  // A = kw / P
  if (r.all || !(kw <= 0.25f * P)) return true;
  const float ax = fabsf(n[0]), ay = fabsf(n[1]), az = fabsf(n[2]);
  const float dn = (fabsf(n[0] * r.dc.x + n[1] * r.dc.y + n[2] * r.dc.z) -
                    (ax * r.dh.x + ay * r.dh.y + az * r.dh.z)) * P;
  // twice the error of the distances is left for cos(angle) >= 0.968 and the roundings here
  const float rl = rho * lambda;
  const float on = (fabsf(n[0] * r.oc.x + n[1] * r.oc.y + n[2] * r.oc.z - h) -
                    (ax * r.oh.x + ay * r.oh.y + az * r.oh.z)) * P;
  const float qn = (fabsf(n[0] * r.qc.x + n[1] * r.qc.y + n[2] * r.qc.z - h) -
                    (ax * r.qh.x + ay * r.qh.y + az * r.qh.z)) * P;
  const float k1 = kw * (1.f / kGrazeNear);
  low = !(dn > r.dir * (k1 + 0x1p-20f * P)) && !(on > rl * (1.05f * k1 + 0x1p-19f * P)) &&
        !(qn > rl * (1.05f * k1 + 0x1p-19f * P) + r.far * (k1 + 0x1p-18f * P));
  return !(dn > r.dir * (kw + 0x1p-20f * P)) && !(on > rl * (1.05f * kw + 0x1p-19f * P)) &&
         !(qn > rl * (1.05f * kw + 0x1p-19f * P) + r.far * (kw + 0x1p-18f * P));
}
// kappa and reach of the triangle, v and edge too; after grazes_plane without `low`.
RT_HD bool grazes_place(const GrazeRays& r, float kappa, float reach, const float* v, float edge,
                        const SearchFrame& f) {
  const float P = pad_grow(kappa) * f.pad + r.extra;
  return !(kGrazeNear * P < 0.5f * (r.dist + reach)) || 
         (comes_near(r, r.oc, r.oh, v, edge + kGrazeNear * P) &&
          comes_near(r, r.qc, r.qh, v, edge + kGrazeNear * P));
}
RT_HD bool grazes(const GrazeRays& r, const GrazeTri& g, const SearchFrame& f) {
  bool low;
  return grazes_plane(r, g.n, g.h, g.kappa, g.lambda, g.reach, f, low) &&
         (low || grazes_place(r, g.kappa, g.reach, g.v, g.edge, f));
}

// A first question, by the angle alone: a triangle's normal and its slope, A for a unit of rho
// without the rays' own pads.
struct GrazeNormal {
  float n[3];
  float slope;  // as kappa: negative infinity for none, infinity for all
};
RT_HD GrazeNormal graze_normal(const GrazeTri& g, const SearchFrame& f) {
  return GrazeNormal{{g.n[0], g.n[1], g.n[2]},
                     g.kappa < 0.f ? -INFINITY
                                   : g.kappa * kGrazeErr / (pad_grow(g.kappa) * f.pad)};
}
// Largest |d| * rho of the rays over the scene, NaN if no bound holds.
RT_HD float graze_steep(const GrazeRays& r, const SearchFrame& f) {
  return r.all ? __builtin_nanf("") : r.dir * (r.dist + f.reach) * (1.f + 0x1p-18f);
}
RT_HD bool grazes_angle(const GrazeRays& r, float steep, const GrazeNormal& g) {
  const float dn = fabsf(g.n[0] * r.dc.x + g.n[1] * r.dc.y + g.n[2] * r.dc.z) -
                   (fabsf(g.n[0]) * r.dh.x + fabsf(g.n[1]) * r.dh.y + fabsf(g.n[2]) * r.dh.z);
  return !(dn > g.slope * steep + 0x1p-19f * r.dir);
}

// The same for one ray, with the triangle's own reach (near_slope: slope * reach): true when the
// ray does not graze it.
RT_HD float graze_near_slope(const GrazeTri& t, const GrazeNormal& g) {
  return t.kappa < 0.f ? -INFINITY : g.slope * t.reach * (1.f + 0x1p-20f);
}
RT_HD void graze_ray(F3 o, F3 d, const SearchFrame& f, float& len, float& dist) {
  const float x = o.x - f.center[0], y = o.y - f.center[1], z = o.z - f.center[2];
  const float most = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
  len = near_sqrt(d.x * d.x + d.y * d.y + d.z * d.z) * (1.f + 0x1p-18f);
  dist = near_sqrt(x * x + y * y + z * z) * (1.f + 0x1p-18f);
  // no bound holds: NaN lets everything through
  if (!(most >= kGrazeDirMin && len <= kGrazeDirMax && dist <= kGrazeHuge)) len = __builtin_nanf("");
}
RT_HD bool graze_clears(const GrazeNormal& g, float near_slope, F3 d, float len, float dist) {
  return fabsf(g.n[0] * d.x + g.n[1] * d.y + g.n[2] * d.z) >
         len * (g.slope * dist + near_slope + 0x1p-19f);
}

// The planes of a cluster of triangles; kappa negative: none can be hit.
struct GrazeCluster {
  float nc[3], hc;  // middle of the normals and of h
  float nh[3], hh;  // half widths
  float kappa, lambda, reach, pad_;  // largest
};
RT_HD void cluster_clear(float* lo, float* hi) {
  for (int k = 0; k < 4; ++k) {
    lo[k] = INFINITY;
    hi[k] = -INFINITY;
  }
}
RT_HD GrazeCluster graze_cluster(const GrazeTri* g, uint32_t n) {
  GrazeCluster c{};
  float lo[4], hi[4];
  cluster_clear(lo, hi);
  c.kappa = -1.f;
  for (uint32_t i = 0; i < n; ++i) {
    if (g[i].kappa < 0.f) continue;
    for (int k = 0; k < 4; ++k) {
      const float x = k < 3 ? g[i].n[k] : g[i].h;
      lo[k] = fminf(lo[k], x);
      hi[k] = fmaxf(hi[k], x);
    }
    c.kappa = fmaxf(c.kappa, g[i].kappa);
    c.lambda = fmaxf(c.lambda, g[i].lambda);
    c.reach = fmaxf(c.reach, g[i].reach);
  }
  if (c.kappa < 0.f) return c;
  for (int k = 0; k < 4; ++k) {
    const float m = 0.5f * (lo[k] + hi[k]), w = fmaxf(hi[k] - m, m - lo[k]) * (1.f + 0x1p-20f);
    (k < 3 ? c.nc[k] : c.hc) = m;
    (k < 3 ? c.nh[k] : c.hh) = w;
  }
  return c;
}
// Never false when grazes_plane is true for one of its triangles.  kappa over its pad grows with
// kappa, so the largest bounds all.
RT_HD bool grazes_cluster(const GrazeRays& r, const GrazeCluster& c, const SearchFrame& f) {
  if (c.kappa < 0.f) return false;
  const float rho = r.dist + c.reach;
  const float P = pad_grow(c.kappa) * f.pad + r.extra, kw = c.kappa * (kGrazeErr * rho);
  if (r.all || !(kw <= 0.25f * P)) return true;
  auto off = [&](const F3& m, const F3& h, float hc, float hh) {
    return (fabsf(c.nc[0] * m.x + c.nc[1] * m.y + c.nc[2] * m.z - hc) -
            (fabsf(c.nc[0]) * h.x + fabsf(c.nc[1]) * h.y + fabsf(c.nc[2]) * h.z +
             c.nh[0] * (fabsf(m.x) + h.x) + c.nh[1] * (fabsf(m.y) + h.y) +
             c.nh[2] * (fabsf(m.z) + h.z) + hh)) * P;
  };
  const float rl = rho * c.lambda;
  return !(off(r.dc, r.dh, 0.f, 0.f) > r.dir * (kw + 0x1p-19f * P)) &&
         !(off(r.oc, r.oh, c.hc, c.hh) > rl * (1.05f * kw + 0x1p-18f * P)) &&
         !(off(r.qc, r.qh, c.hc, c.hh) > rl * (1.05f * kw + 0x1p-18f * P) +
                                             r.far * (kw + 0x1p-17f * P));
}

// ---------------------------------------------------------------------------------------
// Ray against the planes of a wide node (SearchFrame units): the parameter of plane g + h of an
// axis (grid cell g, FP16 offset h) is g * ih + c + h * ih with ih = unit / d and c =
// (base - o) / d.  c is widened outward (down to cn for near planes, up to cf for far ones) by
// the ray's own pad (ray_pad) and by kOffSlack, which covers its own rounding and that of the
// sums; the scale h * ih + ... rounds once more, which kSlack covers on the far side.
struct SlabRay {
  F3 ih, cn, cf;
};
RT_HD void slab_axis(float o, float d, float base, float unit, float pad, float& ih, float& cn,
                     float& cf) {
  // zero components become tiny ones, so the slab of that axis is (almost) the whole line when
  // the origin is inside it and empty otherwise
  const float inv = 1.0f / (fabsf(d) < 0x1p-80f ? (d < 0.f ? -0x1p-80f : 0x1p-80f) : d);
  const float c = (base - o) * inv, w = fabsf(c) * kOffSlack + pad * fabsf(inv);
  ih = inv * unit;
  cn = c - w;
  cf = c + w;
}
RT_HD SlabRay slab_ray(F3 o, F3 d, const SearchFrame& f) {
  SlabRay s;
  const float x = o.x - f.center[0], y = o.y - f.center[1], z = o.z - f.center[2];
  const float pad = ray_pad(sqrtf(x * x + y * y + z * z), f);
  slab_axis(o.x, d.x, f.base[0], f.unit, pad, s.ih.x, s.cn.x, s.cf.x);
  slab_axis(o.y, d.y, f.base[1], f.unit, pad, s.ih.y, s.cn.y, s.cf.y);
  slab_axis(o.z, d.z, f.base[2], f.unit, pad, s.ih.z, s.cn.z, s.cf.z);
  return s;
}

typedef _Float16 rt_h2 __attribute__((ext_vector_type(2)));
// Child c's FP16 plane of a packed quadruple (two words).
RT_HD float plane(uint32_t w01, uint32_t w23, int c) {
  const rt_h2 h = __builtin_bit_cast(rt_h2, c < 2 ? w01 : w23);
  return (float)h[c & 1];
}

// Sort keys of a node's children (its words nx, ny, nz, nm) for a ray whose interval is
// [tlo, thi]: the child's entry parameter, the child in the low two bits; kNoChild, which sorts
// last, for a child that the ray misses or that is absent (only the order of the visits depends
// on the lost bits).
constexpr uint32_t kNoChild = 0xffffffffu;
RT_HD void node_keys(uint4 nx, uint4 ny, uint4 nz, uint4 nm, const SlabRay& sr, float tlo,
                     float thi, uint32_t (&key)[4]) {
  const float gx = (float)(nm.x & 255u), gy = (float)((nm.x >> 8) & 255u),
              gz = (float)((nm.x >> 16) & 255u);
  // plane parameters of the cell's corner; near and far plane words by the ray's sign
  const F3 an = {fmaf(gx, sr.ih.x, sr.cn.x), fmaf(gy, sr.ih.y, sr.cn.y),
                 fmaf(gz, sr.ih.z, sr.cn.z)};
  const F3 af = {fmaf(gx, sr.ih.x, sr.cf.x), fmaf(gy, sr.ih.y, sr.cf.y),
                 fmaf(gz, sr.ih.z, sr.cf.z)};
  const bool sx = sr.ih.x < 0.f, sy = sr.ih.y < 0.f, sz = sr.ih.z < 0.f;
  const uint32_t nx0 = sx ? nx.z : nx.x, nx1 = sx ? nx.w : nx.y, fx0 = sx ? nx.x : nx.z,
                 fx1 = sx ? nx.y : nx.w;
  const uint32_t ny0 = sy ? ny.z : ny.x, ny1 = sy ? ny.w : ny.y, fy0 = sy ? ny.x : ny.z,
                 fy1 = sy ? ny.y : ny.w;
  const uint32_t nz0 = sz ? nz.z : nz.x, nz1 = sz ? nz.w : nz.y, fz0 = sz ? nz.x : nz.z,
                 fz1 = sz ? nz.y : nz.w;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float tn = fmaxf(fmaxf(fmaf(plane(nx0, nx1, c), sr.ih.x, an.x),
                                 fmaf(plane(ny0, ny1, c), sr.ih.y, an.y)),
                           fmaf(plane(nz0, nz1, c), sr.ih.z, an.z));
    const float tf = fminf(fminf(fmaf(plane(fx0, fx1, c), sr.ih.x, af.x),
                                 fmaf(plane(fy0, fy1, c), sr.ih.y, af.y)),
                           fmaf(plane(fz0, fz1, c), sr.ih.z, af.z));
    const float en = fmaxf(tn, tlo);
    const bool hit = (uint32_t)c < nm.w && en <= fminf(fmaf(fabsf(tf), kSlack, tf), thi);
    key[c] = hit ? (__builtin_bit_cast(uint32_t, en) & ~3u) | (uint32_t)c : kNoChild;
  }
}

}  // namespace rti
