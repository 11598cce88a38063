// box_test.h -- the ray / box tests of the traversal, host and device code
// (the host compiles it in tests only).
//
// Every node test of every layout is the reference's slab test
// (wavefront_compute/geometry/mod.rs:44-64): t = (plane - origin) * (1 / dir),
// both operations rounded.  The rounding is monotone in the plane, so a box
// passes whenever a box inside it does, and which triangles a ray can reach is
// decided by their leaf's box alone: the layouts with exact boxes (child
// pairs, child quads) report a hit for the same rays.  A fused t = plane * inv -
// origin * inv would take half the instructions, but its error is relative to
// origin * inv and not to the distance: it loses boxes that the slab test
// passes where the origin is small against the plane.
#ifndef RDRT_BOX_TEST_H
#define RDRT_BOX_TEST_H

#include <math.h>
#include <stdint.h>

#ifdef __HIP__
#include <hip/hip_runtime.h>
#define RDRT_BOX_FN __host__ __device__ __forceinline__
#pragma clang fp contract(off)
#else
#define RDRT_BOX_FN inline
#endif

namespace rdrt {
namespace {

struct F3 {
  float x, y, z;
};

// Ray/AABB slab test (wavefront_compute/geometry/mod.rs:44-64).  inv_d is
// 1/dir, hoisted out of the node loop; the per-node values are unchanged.
[[maybe_unused]] RDRT_BOX_FN bool slab(F3 o, F3 inv_d, float tmin, float tmax, float mnx, float mny, float mnz,
                                       float mxx, float mxy, float mxz, float &tnear) {
  float t0x = (mnx - o.x) * inv_d.x, t0y = (mny - o.y) * inv_d.y, t0z = (mnz - o.z) * inv_d.z;
  float t1x = (mxx - o.x) * inv_d.x, t1y = (mxy - o.y) * inv_d.y, t1z = (mxz - o.z) * inv_d.z;
  float nx = fminf(t0x, t1x), ny = fminf(t0y, t1y), nz = fminf(t0z, t1z);
  float fx = fmaxf(t0x, t1x), fy = fmaxf(t0y, t1y), fz = fmaxf(t0z, t1z);
  float tn = fmaxf(fmaxf(nx, ny), nz);
  float tf = fminf(fminf(fx, fy), fz);
  tnear = tn;
  return tn <= tf && tmin < tf && tn < tmax;
}

// A ray as the node tests take it.  plain: origin and 1 / dir are finite and
// 1 / dir is not zero, so that the direction's sign alone tells the near
// plane of an axis from the far one; otherwise a product may be NaN, which
// drops out of the slab test's min and max.
struct RayBox {
  F3 o, inv;
  bool plain;
};
[[maybe_unused]] RDRT_BOX_FN RayBox ray_box(F3 o, F3 inv) {
  const auto finite = [](float v) { return fabsf(v) < (float)INFINITY; };
  const auto proper = [&](float v) { return finite(v) && v != 0.0f; };
  return RayBox{o, inv, finite(o.x) && finite(o.y) && finite(o.z) && proper(inv.x) && proper(inv.y) && proper(inv.z)};
}

// The slab test of a box whose near and far planes (n, f) were chosen by the
// direction's sign; PLAIN leaves out the min and max that choose them.
template <bool PLAIN>
RDRT_BOX_FN bool planes_hit(const RayBox &r, float tmin, float tmax, float nx, float ny, float nz, float fx, float fy,
                            float fz, float &tnear) {
  float ax = (nx - r.o.x) * r.inv.x, ay = (ny - r.o.y) * r.inv.y, az = (nz - r.o.z) * r.inv.z;
  float bx = (fx - r.o.x) * r.inv.x, by = (fy - r.o.y) * r.inv.y, bz = (fz - r.o.z) * r.inv.z;
  if (!PLAIN) {
    const float cx = ax, cy = ay, cz = az;
    ax = fminf(cx, bx), ay = fminf(cy, by), az = fminf(cz, bz);
    bx = fmaxf(cx, bx), by = fmaxf(cy, by), bz = fmaxf(cz, bz);
  }
  const float tn = fmaxf(fmaxf(ax, ay), az), tf = fminf(fminf(bx, by), bz);
  tnear = tn;
  return tn <= tf && tmin < tf && tn < tmax;
}

// Byte c of a quantized node word, decoded as the host that chose it does:
// corner + q * step, rounded once (q * step is exact, so one fused operation
// gives the same value).
[[maybe_unused]] RDRT_BOX_FN float dequant(float corner, uint32_t word, int c, float step) {
  return __builtin_fmaf((float)((word >> (8 * c)) & 0xffu), step, corner);
}

}  // namespace
}  // namespace rdrt

#endif
