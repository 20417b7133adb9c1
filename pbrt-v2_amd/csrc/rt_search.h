// rt_search.h -- a ray against the nodes of the per-ray path's search tree (RhItem::snode, see
// rt_internal.h), for the per-ray kernel and for host code that walks the same tree.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace rti {

#define RT_HD __host__ __device__ __forceinline__

constexpr float kSlack = 0x1p-16f;     // relative slack of the slab-test parameters
constexpr float kOffSlack = 0x1p-20f;  // the same of a ray's plane offsets

struct F3 {
  float x, y, z;
};

// Ray against the planes of a wide node (SearchFrame units): the parameter of plane g + h of an
// axis (grid cell g, FP16 offset h) is g * ih + c + h * ih with ih = unit / d and c =
// (base - o) / d.  c is widened outward (down to cn for near planes, up to cf for far ones) by
// kOffSlack, which covers its own rounding and that of the sums; the scale h * ih + ... rounds
// once more, which kSlack covers on the far side.
struct SlabRay {
  F3 ih, cn, cf;
};
RT_HD void slab_axis(float o, float d, float base, float unit, float& ih, float& cn, float& cf) {
  // zero components become tiny ones, so the slab of that axis is (almost) the whole line when
  // the origin is inside it and empty otherwise
  const float inv = 1.0f / (fabsf(d) < 0x1p-80f ? (d < 0.f ? -0x1p-80f : 0x1p-80f) : d);
  const float c = (base - o) * inv, w = fabsf(c) * kOffSlack;
  ih = inv * unit;
  cn = c - w;
  cf = c + w;
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
