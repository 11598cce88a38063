// trace_device.h -- device code of the closest-hit traversal kernels for
// gfx950 (wave64), shared by the translation units that instantiate them.
//
// Two kernels share one result definition, that of the reference CPU
// traversal (shader/ray-tracing/src/backend/wavefront_compute/geometry/naive/
// traverse_cpu.rs:52-245): the last accepted triangle wins, a triangle is
// accepted when its t lies in [t_min, far] of the ray range in object space
// (wavefront_compute/geometry/mod.rs:104-155), and far shrinks to each accepted
// hit.
//
//  * k_trace_ref walks the reference's 48-byte forest by its stackless
//    hit/miss links (traverse_cpu.rs:283-319) in the reference order, with the
//    reference's per-test arithmetic; its hits and visit counters equal the
//    oracle's bit for bit.
//  * The fast kernels walk child-pair or child-quad layouts of a tree of
//    their own front to back, with a per-lane stack in LDS (column layout
//    [entry][lane]: each lane owns one bank at every depth, so stack traffic
//    is conflict-free), and test triangles from 64-byte pre-pass records with
//    the reference's arithmetic, so t, u, v are bit-identical.  Their box tests
//    are the reference's too (box_test.h), so child pairs and child quads,
//    which hold the same leaf boxes, report a hit for the same rays, and only
//    the visit order differs, which can change the winner among hits with
//    equal t.  Quantized quads widen the boxes to 8-bit planes: a ray that
//    passes a leaf's box by less than a plane's step may hit with them only.
//
//    What bounded these kernels was idle lanes: with every lane doing whatever
//    it was at, 9 (1M rays in 100k triangles) to 15 (height field, first
//    bounce) of 64 lanes worked per vector instruction.  trace_wave gives the
//    wave one kind of work at a time and refills it.  With near and far planes
//    chosen by the loads, no round trip to memory behind the node tests and a
//    work counter per XCD, 1M rays went from 0.49 to 0.35 ms, the 1080p frame
//    from 2.4 to 1.8 ms, a height-field step of 16 views from 24.7 to 20.8 ms,
//    a batch of 16 scenes from 4.3 to 2.4 ms.  (A fused multiply-add per plane
//    would make that 0.33, 1.7 and 2.3 ms, but it loses hits: box_test.h.)
//
// Compiled with -ffp-contract=off and IEEE division/sqrt: one rounding per
// operation, as in the reference.
#ifndef RDRT_TRACE_DEVICE_H
#define RDRT_TRACE_DEVICE_H

#include <algorithm>
#include <type_traits>

#include "box_test.h"
#include "trace_kernels.h"

#pragma clang fp contract(off)

namespace rdrt {
namespace {

constexpr uint32_t F_FORCE_OPAQUE = 0x01, F_FORCE_NON_OPAQUE = 0x02, F_END_SEARCH = 0x04, F_CULL_BACK = 0x10,
                   F_CULL_FRONT = 0x20, F_CULL_OPAQUE = 0x40, F_CULL_NON_OPAQUE = 0x80,
                   F_SKIP_TRIANGLES = 0x100, F_FLIP = 0x400;
constexpr uint32_t GI_CULL_DISABLE = 0x1, GI_FLIP = 0x2, GI_FORCE_OPAQUE = 0x4, GI_FORCE_NO_OPAQUE = 0x8;

__device__ __forceinline__ F3 f3(float x, float y, float z) { return F3{x, y, z}; }
__device__ __forceinline__ F3 sub(F3 a, F3 b) { return f3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ float dot(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ F3 cross(F3 a, F3 b) {
  return f3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ F3 normalize(F3 a) {
  float m = dot(a, a);
  if (m > 0.0f) {
    float inv = 1.0f / sqrtf(m);
    return f3(a.x * inv, a.y * inv, a.z * inv);
  }
  return a;
}
__device__ __forceinline__ F3 recip(F3 a) { return f3(1.0f / a.x, 1.0f / a.y, 1.0f / a.z); }

// Triangle test given the vertex-only quantities (geometry/mod.rs:118-154).
// b == 0 is a miss.
__device__ __forceinline__ bool tri_core(F3 o, F3 d, float rn, float rf, F3 v0, F3 e1, F3 e2, F3 n, float uu,
                                         float uv, float vv, float inverse_d, bool cull_enable, bool cull_back,
                                         float &t, float &u, float &v, bool &back) {
  float b = dot(n, d);
  if (b == 0.0f) return false;
  if (cull_enable && cull_back == (b < 0.0f)) return false;
  F3 w0 = sub(o, v0);
  float a = -dot(n, w0);
  float tt = a / b;
  if (tt < rn || tt > rf) return false;
  F3 p = f3(o.x + tt * d.x, o.y + tt * d.y, o.z + tt * d.z);
  F3 w = sub(p, v0);
  float wu = dot(w, e1);
  float wv = dot(w, e2);
  float uu_ = (uv * wv - vv * wu) * inverse_d;
  if (uu_ < 0.0f || uu_ > 1.0f) return false;
  float vv_ = (uv * wu - uu * wv) * inverse_d;
  if (vv_ < 0.0f || (uu_ + vv_) > 1.0f) return false;
  t = tt;
  u = uu_;
  v = vv_;
  back = b < 0.0f;
  return true;
}

// flag.rs:30-75
__device__ __forceinline__ uint32_t merge_flags(uint32_t f, uint32_t gi) {
  if (gi & GI_CULL_DISABLE) f &= ~(F_CULL_BACK | F_CULL_FRONT);
  if (gi & GI_FLIP) f ^= F_FLIP;
  if (gi & GI_FORCE_OPAQUE) f |= F_FORCE_OPAQUE;
  if (gi & GI_FORCE_NO_OPAQUE) f |= F_FORCE_NON_OPAQUE;
  return f;
}
// flag.rs:78-91.  Opaque for this ray: the geometry's flag, forced either way by the merged
// ray / instance flags (flag.rs cull_geometry).
__device__ __forceinline__ bool geometry_opaque(uint32_t f, uint32_t gflags) {
  return ((gflags & RDRT_GEOMETRY_FLAG_OPAQUE) || (f & F_FORCE_OPAQUE)) && !(f & F_FORCE_NON_OPAQUE);
}
// Any-hit behaviour of a hit on global triangle `tri` (traverse_cpu.rs:
// 164-185): an opaque hit commits; a non-opaque one takes the caller's
// per-triangle behaviour, or is accepted without a table.
__device__ __forceinline__ uint32_t anyhit_behavior(const TraceParams &p, bool opaque, uint32_t tri) {
  return (opaque || !p.anyhit) ? RDRT_ANYHIT_ACCEPT : (uint32_t)p.anyhit[tri];
}
__device__ __forceinline__ bool geometry_passes(uint32_t f, uint32_t gflags) {
  bool opaque = geometry_opaque(f, gflags);
  return (opaque && !(f & F_CULL_OPAQUE)) || (!opaque && !(f & F_CULL_NON_OPAQUE));
}
// flag.rs:94-105
__device__ __forceinline__ void cull_triangle(uint32_t f, bool &enable, bool &back) {
  bool flip = f & F_FLIP, cf = f & F_CULL_FRONT, cb = f & F_CULL_BACK;
  enable = cf || cb;
  back = (flip && cb) || (!flip && cf);
}

// Object-space ray of an instance (traverse_cpu.rs:99-104): inverse transform
// of the origin with the w divide, 3x3 part on the direction, scaling = its
// length, direction normalized.
__device__ __forceinline__ void object_ray(const float *m, F3 o, F3 d, F3 &bo, F3 &bd, float &scaling) {
  float x = o.x * m[0] + o.y * m[4] + o.z * m[8] + 1.0f * m[12];
  float y = o.x * m[1] + o.y * m[5] + o.z * m[9] + 1.0f * m[13];
  float z = o.x * m[2] + o.y * m[6] + o.z * m[10] + 1.0f * m[14];
  float w = o.x * m[3] + o.y * m[7] + o.z * m[11] + 1.0f * m[15];
  bo = f3(x / w, y / w, z / w);
  F3 dd = f3(d.x * m[0] + d.y * m[4] + d.z * m[8], d.x * m[1] + d.y * m[5] + d.z * m[9],
             d.x * m[2] + d.y * m[6] + d.z * m[10]);
  scaling = sqrtf(dot(dd, dd));
  bd = normalize(dd);
}

struct RayIn {
  F3 o, d;
  float tmin, tmax;
  uint32_t flags, mask, tlas_idx;
};

__device__ __forceinline__ RayIn load_ray(const TraceParams &p, uint32_t rid) {
  const float4 *rp = reinterpret_cast<const float4 *>(p.rays + rid);
  float4 a = rp[0], b = rp[1];
  RayIn r;
  r.o = f3(a.x, a.y, a.z);
  r.tmin = a.w;
  r.d = f3(b.x, b.y, b.z);
  r.tmax = b.w;
  r.flags = p.flags;
  r.mask = p.cull_mask;
  r.tlas_idx = p.tlas_idx;
  if (p.meta) {
    uint4 m = *reinterpret_cast<const uint4 *>(p.meta + rid);
    r.flags = m.x;
    r.mask = m.y;
    r.tlas_idx = m.z;
  }
  return r;
}

// Root of the TLAS bound at tlas_idx, or null when unbound / deleted.
__device__ __forceinline__ const TlasRoot *bound_root(const TraceParams &p, uint32_t tlas_idx) {
  if (tlas_idx >= p.nbinding) return nullptr;
  uint32_t th = p.binding[tlas_idx];
  if (th >= p.ntlas) return nullptr;
  const TlasRoot *r = p.tlas_roots + th;
  return r->ref_root == kInvalid ? nullptr : r;
}

struct Best {
  uint32_t k = kInvalid;  // triangle slot (redirect index)
  uint32_t geo = 0, inst = 0;
  float t = 0.0f, u = 0.0f, v = 0.0f;
  bool back = false;
};

// ids maps best.k to the global triangle: p.tri_ids (fast) or p.redirect (reference).
__device__ __forceinline__ void write_result(const TraceParams &p, const uint32_t *ids, uint32_t rid,
                                             const Best &best, uint32_t cn, uint32_t ct, uint32_t ci) {
  uint4 h = make_uint4(RDRT_MISS, 0u, 0u, 0u);
  uint4 hm = make_uint4(RDRT_MISS, RDRT_MISS, 0u, RDRT_MISS);
  if (best.k != kInvalid) {
    const GeoRec &g = p.geos[best.geo];
    h.x = ids[best.k] - g.primitive_start;
    h.y = __float_as_uint(best.t);
    h.z = __float_as_uint(best.u);
    h.w = __float_as_uint(best.v);
    if (p.hit_meta) {
      const InstRec &in = p.insts[best.inst];
      hm = make_uint4(g.geometry_idx, in.order, best.back ? RDRT_HIT_KIND_BACK_FACING_TRIANGLE
                                                          : RDRT_HIT_KIND_FRONT_FACING_TRIANGLE,
                      in.custom_index);
    }
  }
  *reinterpret_cast<uint4 *>(p.hits + rid) = h;
  if (p.hit_meta) *reinterpret_cast<uint4 *>(p.hit_meta + rid) = hm;
  if (p.hitx) p.hitx[rid] = make_uint2(best.geo, best.inst);
  if (p.counters) {
    p.counters[3 * rid + 0] = cn;
    p.counters[3 * rid + 1] = ct;
    p.counters[3 * rid + 2] = ci;
  }
}

// Blocks are dispatched round-robin over the 8 XCDs (each with its own L2).
// Remap the first `used` physical blocks so each XCD works on one contiguous
// range of rays: neighbouring (coherent) rays then share an L2.
__device__ __forceinline__ uint32_t xcd_block(uint32_t i, uint32_t used) {
  const uint32_t xcd = i % 8u, local = i / 8u, per = used / 8u, rem = used % 8u;
  return xcd < rem ? xcd * (per + 1u) + local : rem * (per + 1u) + (xcd - rem) * per + local;
}

// Inner-node tests of the fast traversal: the children of one node that the
// ray meets, in `r[0 .. n)`, farthest first (what follows r[n - 1] is
// undefined).
struct Kids {
  uint32_t n, r[4];
};

__device__ __forceinline__ bool negative(float v) { return (__float_as_uint(v) & 0x80000000u) != 0u; }

__device__ __forceinline__ Kids kids_pair(const PairNode *node, const RayBox &r, float tmin, float tmax) {
  const float4 *q = reinterpret_cast<const float4 *>(node);
  const float4 a = q[0], b = q[1], c = q[2], d = q[3];
  float tl, tr;
  const bool hl = slab(r.o, r.inv, tmin, tmax, a.x, a.y, a.z, b.x, b.y, b.z, tl);
  const bool hr = slab(r.o, r.inv, tmin, tmax, c.x, c.y, c.z, d.x, d.y, d.z, tr);
  const uint32_t lref = __float_as_uint(a.w), rref = __float_as_uint(c.w);
  const bool rlast = hr && (!hl || tr < tl);  // the right child is the nearest hit
  Kids k;
  k.n = (uint32_t)hl + (uint32_t)hr;
  const uint32_t near_ref = rlast ? rref : lref, far_ref = rlast ? lref : rref;
  k.r[0] = k.n == 2u ? far_ref : near_ref;
  k.r[1] = near_ref;
  k.r[2] = k.r[3] = 0u;
  return k;
}

// Sort key of one quad child: a double whose high word is the entry distance
// and whose low word is the child's ref, 0 when missed.  Distances are
// clamped to at least 2^-100, so every hit is a positive normal double (its
// float bits are below those of infinity) and the order of the doubles is the
// order of the distances.
__device__ __forceinline__ double quad_key(bool hit, float tnear, uint32_t ref) {
  const uint32_t hi = hit ? __float_as_uint(fmaxf(tnear, 7.88860905e-31f)) : 0u;
  return __hiloint2double((int)hi, (int)ref);
}
// One compare-exchange in two instructions (fmin / fmax on values that the
// compiler cannot prove to be no signaling NaN take four).
__device__ __forceinline__ void order2(double &a, double &b) {
  double hi, lo;
  asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
  asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
  a = hi;
  b = lo;
}
__device__ __forceinline__ Kids sort_kids(const bool h[4], const float t[4], uint4 rf) {
  double k0 = quad_key(h[0], t[0], rf.x), k1 = quad_key(h[1], t[1], rf.y), k2 = quad_key(h[2], t[2], rf.z),
         k3 = quad_key(h[3], t[3], rf.w);
  // sorting network of four: hits descend by entry distance, misses last
  order2(k0, k1);
  order2(k2, k3);
  order2(k0, k2);
  order2(k1, k3);
  order2(k1, k2);
  Kids k;
  k.n = (uint32_t)h[0] + (uint32_t)h[1] + (uint32_t)h[2] + (uint32_t)h[3];
  k.r[0] = (uint32_t)__double2loint(k0);
  k.r[1] = (uint32_t)__double2loint(k1);
  k.r[2] = (uint32_t)__double2loint(k2);
  k.r[3] = (uint32_t)__double2loint(k3);
  return k;
}

template <bool PLAIN>
__device__ __forceinline__ Kids kids_quad(const QuadNode *node, const RayBox &r, float tmin, float tmax) {
  // the rows of the near and the far planes of an axis swap with the
  // direction's sign: 16 bytes apart, so the loads pick them
  const char *q = reinterpret_cast<const char *>(node);
  const uint32_t sx = (__float_as_uint(r.inv.x) >> 27) & 16u, sy = (__float_as_uint(r.inv.y) >> 27) & 16u,
                 sz = (__float_as_uint(r.inv.z) >> 27) & 16u;
  const float4 xn = *reinterpret_cast<const float4 *>(q + sx), xf = *reinterpret_cast<const float4 *>(q + (sx ^ 16u));
  const float4 yn = *reinterpret_cast<const float4 *>(q + 32 + sy),
               yf = *reinterpret_cast<const float4 *>(q + 32 + (sy ^ 16u));
  const float4 zn = *reinterpret_cast<const float4 *>(q + 64 + sz),
               zf = *reinterpret_cast<const float4 *>(q + 64 + (sz ^ 16u));
  const uint4 rf = *reinterpret_cast<const uint4 *>(q + 96);
  float t[4];
  bool h[4];
  h[0] = planes_hit<PLAIN>(r, tmin, tmax, xn.x, yn.x, zn.x, xf.x, yf.x, zf.x, t[0]);
  h[1] = planes_hit<PLAIN>(r, tmin, tmax, xn.y, yn.y, zn.y, xf.y, yf.y, zf.y, t[1]);  // slots 0, 1 always used
  h[2] = planes_hit<PLAIN>(r, tmin, tmax, xn.z, yn.z, zn.z, xf.z, yf.z, zf.z, t[2]) && rf.z != kInvalid;
  h[3] = planes_hit<PLAIN>(r, tmin, tmax, xn.w, yn.w, zn.w, xf.w, yf.w, zf.w, t[3]) && rf.w != kInvalid;
  return sort_kids(h, t, rf);
}

template <bool PLAIN>
__device__ __forceinline__ Kids kids_qquad(const QuadNodeQ *node, const RayBox &r, float tmin, float tmax) {
  const float4 *q = reinterpret_cast<const float4 *>(node);
  const float4 a = q[0];                                  // corner, x step
  const uint4 rf = *reinterpret_cast<const uint4 *>(q + 1);
  const uint4 xy = *reinterpret_cast<const uint4 *>(q + 2);  // lox, hix, loy, hiy
  const float4 zs = q[3];                                 // loz, hiz (bits), y step, z step
  const uint32_t loz = __float_as_uint(zs.x), hiz = __float_as_uint(zs.y);
  const bool sx = negative(r.inv.x), sy = negative(r.inv.y), sz = negative(r.inv.z);
  const uint32_t nx = sx ? xy.y : xy.x, fx = sx ? xy.x : xy.y, ny = sy ? xy.w : xy.z, fy = sy ? xy.z : xy.w,
                 nz = sz ? hiz : loz, fz = sz ? loz : hiz;
  float t[4];
  bool h[4];
#pragma unroll
  for (int c = 0; c < 4; c++)
    h[c] = planes_hit<PLAIN>(r, tmin, tmax, dequant(a.x, nx, c, a.w), dequant(a.y, ny, c, zs.z),
                             dequant(a.z, nz, c, zs.w), dequant(a.x, fx, c, a.w), dequant(a.y, fy, c, zs.z),
                             dequant(a.z, fz, c, zs.w), t[c]);
  h[2] = h[2] && rf.z != kInvalid;  // slots 0, 1 always used
  h[3] = h[3] && rf.w != kInvalid;
  return sort_kids(h, t, rf);
}

template <int LAYOUT, bool PLAIN>
__device__ __forceinline__ Kids test_kids(const TraceParams &p, bool world, uint32_t ref, const RayBox &r, float tmin,
                                          float tmax) {
  if constexpr (LAYOUT == 2) return kids_qquad<PLAIN>((world ? p.tlas_qquads : p.tri_qquads) + ref, r, tmin, tmax);
  else if constexpr (LAYOUT == 1) return kids_quad<PLAIN>((world ? p.tlas_quads : p.tri_quads) + ref, r, tmin, tmax);
  else return kids_pair((world ? p.tlas_pairs : p.tri_pairs) + ref, r, tmin, tmax);
}

// A lane's traversal stack: the first R entries in LDS (column layout:
// entry i of the lane at lds[i * B], its own bank at every depth), deeper
// ones (rare) in the lane's private memory.  It holds up to S node refs and
// two end marks.  A step writes its (up to) three farther children at the
// top without asking how many there are and reads the entry below before its
// node arrives, so neither branches nor a second round trip to memory follow
// the box tests.
template <int K, int S, int B>
struct LaneStack {
  static constexpr uint32_t R = K + 4, N = S + 2, kSpill = N > R ? N - R : 1, kRows = R + 6;
  uint32_t *lds;
  // kSpill words of private memory: an array of its own (inside, it would keep sp in memory too) and volatile (else the
  // compiler turns it into registers that it indexes in loops)
  volatile uint32_t *spill;
  uint32_t *status;
  uint32_t sp;

  // the object-space ray of the lane's instance, for the triangle tests, in
  // the six LDS rows above the stack (the node tests need only the RayBox)
  __device__ __forceinline__ void set_ray(F3 o, F3 d) {
    float *q = reinterpret_cast<float *>(lds + R * B);
    q[0] = o.x, q[B] = o.y, q[2 * B] = o.z, q[3 * B] = d.x, q[4 * B] = d.y, q[5 * B] = d.z;
  }
  __device__ __forceinline__ void get_ray(F3 &o, F3 &d) const {
    const float *q = reinterpret_cast<const float *>(lds + R * B);
    o = f3(q[0], q[B], q[2 * B]);
    d = f3(q[3 * B], q[4 * B], q[5 * B]);
  }
  // near the end of the LDS rows, or of the stack: put() spills, or drops and reports
  __device__ __forceinline__ bool deep() const { return sp + 3u > (R < N ? R : N); }
  __device__ __forceinline__ uint32_t get(uint32_t i) const {
    if (N <= R || i < R) return lds[i * B];
    uint32_t v = spill[i - R];
    asm volatile("" : "+v"(v));  // keeps the two loads apart: one load through a selected pointer would be a flat one
    return v;
  }
  __device__ __forceinline__ void put(uint32_t i, uint32_t v) {
    if (i < (N < R ? N : R)) lds[i * B] = v;
    else if (i < N) spill[i - R] = v;
    else atomicOr(status, 1u);  // unreachable when S covers the built depth
  }
  __device__ __forceinline__ void push(uint32_t v) {
    put(sp, v);
    if (sp < N) sp++;
  }
  __device__ __forceinline__ uint32_t pop() { return get(--sp); }

  // The step of a lane at an inner node: kids() tests the node; returns the
  // nearest child hit, or the top of the stack when none is.
  template <int LAYOUT, class F>
  __device__ __forceinline__ uint32_t step(F &&kids) {
    const bool slow = __ballot(deep()) != 0ull;  // wave-uniform, rare
    const uint32_t top = slow ? get(sp - 1u) : lds[(sp - 1u) * B];
    const Kids k = kids();
    if (slow) {
      for (uint32_t j = 0; j + 1u < k.n; j++) put(sp + j, j == 0u ? k.r[0] : j == 1u ? k.r[1] : k.r[2]);
    } else {
      uint32_t *at = lds + sp * B;
      at[0] = k.r[0];
      if constexpr (LAYOUT != 0) {
        at[B] = k.r[1];
        at[2 * B] = k.r[2];
      }
    }
    sp = min(sp + k.n - 1u, N);
    uint32_t r = k.n == 1u ? k.r[0] : top;
    r = k.n == 2u ? k.r[1] : r;
    if constexpr (LAYOUT != 0) {
      r = k.n == 3u ? k.r[2] : r;
      r = k.n == 4u ? k.r[3] : r;
    }
    return r;
  }
};

// ------------------------------------------------------------------------
// Fast kernel: front-to-back traversal, one ray per lane, one kind of work
// per wave step.
//
// A lane is at an inner node, at a leaf of triangles, or at the TLAS (a leaf
// of instances, or a BLAS it has finished).  Each wave step does the work that
// enough lanes wait for, the others keep their place: an inner step serves
// TLAS and BLAS alike (the lane's current ray is the world or the object
// ray), a leaf step tests all triangles of the leaf.  A loop in which every
// lane does whatever it is at runs all three bodies for a few lanes each.
// ------------------------------------------------------------------------
constexpr uint32_t kRefExit = 0x7ffffff0u;  // the lane's BLAS is exhausted
constexpr uint32_t kRefDone = 0x7ffffff1u;  // the lane's ray is finished (or it has none)
// lane status bits
constexpr uint32_t kStOpaque = 1u, kStCull = 2u, kStCullBack = 4u, kStEnd = 8u, kStSecond = 16u, kStBack = 32u,
                   kStWorld = 64u, kStGeometries = 128u;  // kStGeometries: geometries of the instance are left to visit
constexpr uint32_t kStMoreShift = 8;                      // instances of the TLAS leaf still to visit

__device__ __forceinline__ uint32_t wave_rank(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// Lanes of the wave for which v holds, as a scalar.
__device__ __forceinline__ uint32_t wave_count(bool v) {
  return __builtin_amdgcn_readfirstlane((uint32_t)__popcll(__ballot(v)));
}

// Traces the slots [next, end) of the launch and every chunk that more(next,
// end) gets after them (false: no more), refilling the wave when kRefill
// lanes are idle (16 and 48 instead of 32: a 1080p frame 0.7 and 1.8 % slower,
// a height-field step 0.5 and 3.0 %).  Slots below n0 belong to the first
// segment.
constexpr uint32_t kRefill = 32;
// Inner steps go on while 1 / kKeep of the busy lanes want them.  Fewer lanes
// waste vector instructions, more hold back the leaves whose hits shorten the
// rays (2, 4 and 8 instead of 3: 1M rays in 100k triangles 3.2, 1.6 and 9.3 %
// slower, a batch of 16 scenes 0.8, 2.8 and 13.8 %, a 1080p frame 0.6, 0.5 and
// 2.4 %).
constexpr uint32_t kKeep = 3;
// Leaves go before instances unless the lanes at instances outnumber those at
// leaves by more than this: an instance step costs twice a leaf's, so it waits
// for company (1 and 5 instead of 3: a material step 0.9 and 0.3 % slower, a
// batch of 16 scenes 2.8 and 1.1 %, a height-field step 1.2 % slower and 0.7 %
// faster).
constexpr uint32_t kLeavesFirst = 3;

template <int K, int S, int B, bool CNT, int LAYOUT, class More>
__device__ __forceinline__ void trace_wave(const TraceParams &p, uint32_t n0, uint32_t next, uint32_t end,
                                           uint32_t *lds, More &&more) {
  volatile uint32_t spill[LaneStack<K, S, B>::kSpill];
  LaneStack<K, S, B> stk{lds, spill, p.status, 1u};
  RayBox box = {};                               // the current ray: world or object space
  float near_ = 0.0f, far_ = 0.0f, s = 1.0f;     // range: [near_, far_ * s] in its space
  uint32_t ref = kRefDone, rid = kInvalid, st = 0u, inst = 0u, geo = 0u;
  uint32_t best_k = kInvalid, best_geo = 0u, best_inst = 0u;
  float best_u = 0.0f, best_v = 0.0f;
  uint32_t cn = 0, ct = 0, ci = 0;
  bool last = false;  // no chunk is left

  auto ray_of = [&]() {
    TraceParams q = p;
    if (st & kStSecond) {
      q.rays = p.rays2;
      q.flags = p.flags2;
    }
    return load_ray(q, rid);
  };

  auto node_step = [&](auto plain) {
    const bool world = (st & kStWorld) != 0u;
    if constexpr (CNT) cn += world ? 0u : 1u;
    const float fs = far_ * s;
    ref = stk.template step<LAYOUT>(
        [&]() { return test_kids<LAYOUT, decltype(plain)::value>(p, world, ref, box, near_, fs); });
  };

  for (;;) {
    const uint32_t idle = wave_count(ref == kRefDone);
    if (idle == 64u || (!last && idle >= kRefill)) {
      if (ref == kRefDone && rid != kInvalid) {
        Best best;
        best.k = best_k;
        best.geo = best_geo;
        best.inst = best_inst;
        best.t = far_;  // far shrinks to each accepted hit
        best.u = best_u;
        best.v = best_v;
        best.back = (st & kStBack) != 0u;
        TraceParams q = p;
        if (st & kStSecond) {
          q.hits = p.hits2;
          q.hitx = p.hitx2;
          q.counters = nullptr;
        }
        write_result(q, p.tri_ids, rid, best, cn, ct, ci);
        rid = kInvalid;
      }
      if (next >= end) {
        if (!last) last = !more(next, end);
        if (last) {
          if (idle == 64u) break;
          continue;
        }
      }
      const uint64_t m = __ballot(ref == kRefDone);
      const uint32_t slot = next + wave_rank(m);
      if (ref == kRefDone && slot < end) {
        const bool second = slot >= n0;
        st = kStWorld | (second ? kStSecond : 0u);
        const uint32_t qs = second ? slot - n0 : slot;
        const uint32_t *queue = second ? p.queue2 : p.queue;
        rid = queue ? queue[qs] : qs;
        if (rid < p.n) {  // a queue entry always names one of the n rays
          const RayIn r = ray_of();
          const F3 winv = recip(r.d);
          box = ray_box(r.o, winv);
          near_ = r.tmin;
          far_ = r.tmax;
          s = 1.0f;
          best_k = kInvalid;
          if constexpr (CNT) cn = ct = ci = 0u;
          const TlasRoot *root = bound_root(p, r.tlas_idx);
          float tn;
          if (root && slab(r.o, winv, near_, far_, root->mn[0], root->mn[1], root->mn[2], root->mx[0], root->mx[1],
                           root->mx[2], tn)) {
            ref = LAYOUT ? p.tlas_quad_roots[root - p.tlas_roots] : root->root_ref;
            stk.lds[0] = kRefDone;  // the end mark of the ray
            stk.sp = 1u;
          }
        } else {
          rid = kInvalid;
        }
      }
      next = min(end, next + idle);
      continue;
    }
    uint32_t a = wave_count(ref < kRefExit);
    if (a * kKeep >= 64u - idle) {
      // the steps leave `box` as it is: which test they take is decided once
      const bool plain = LAYOUT == 0 || __ballot(ref < kRefExit && !box.plain) == 0ull;
      if (plain) {
        do {
          if (ref < kRefExit) node_step(std::true_type{});
          a = wave_count(ref < kRefExit);
        } while (a * kKeep >= 64u - idle);
      } else {
        do {
          if (ref < kRefExit) node_step(std::false_type{});
          a = wave_count(ref < kRefExit);
        } while (a * kKeep >= 64u - idle);
      }
      continue;
    }
    const bool leaf = (ref & kLeafBit) != 0u, world = (st & kStWorld) != 0u;
    if (kLeavesFirst * wave_count(leaf && !world) >= wave_count(ref == kRefExit || (leaf && world))) {
      if (leaf && !world) {
        const uint32_t k0 = (ref & ~kLeafBit) >> kLeafCountBits, k1 = k0 + (ref & kLeafMaxCount);
        F3 o, bd;
        stk.get_ray(o, bd);
        ref = stk.get(stk.sp - 1u);
        for (uint32_t k = k0; k < k1; k++) {
          if constexpr (CNT) ct++;
          const float4 *q = reinterpret_cast<const float4 *>(p.tris + k);
          const float4 ta = q[0], tb = q[1], tc = q[2], td = q[3];
          float t, u, v;
          bool back;
          if (tri_core(o, bd, near_, far_ * s, f3(ta.x, ta.y, ta.z), f3(tb.x, tb.y, tb.z), f3(tc.x, tc.y, tc.z),
                       f3(td.x, td.y, td.z), ta.w, tb.w, tc.w, td.w, (st & kStCull) != 0u, (st & kStCullBack) != 0u, t,
                       u, v, back)) {
            uint32_t beh = (st & kStOpaque) ? RDRT_ANYHIT_ACCEPT : anyhit_behavior(p, false, p.tri_ids[k]);
            if (beh & RDRT_ANYHIT_ACCEPT) {
              far_ = t / s;
              best_k = k;
              best_geo = geo;
              best_inst = inst;
              best_u = u;
              best_v = v;
              st = back ? st | kStBack : st & ~kStBack;
              if (st & kStEnd) beh |= RDRT_ANYHIT_END_SEARCH;
            }
            if (beh & RDRT_ANYHIT_END_SEARCH) {
              ref = kRefDone;
              break;
            }
          }
        }
        stk.sp--;
      }
    } else if (ref == kRefExit || (leaf && world)) {
      // the next geometry of the lane's instance, or the next instance of its
      // TLAS leaf, that the ray may hit; back to the TLAS when there is none
      const RayIn r = ray_of();
      const F3 winv = recip(r.d);
      uint32_t left, g, gend, fl;
      F3 o = r.o, inv = winv;  // the object ray of the instance
      if (world) {
        inst = ((ref & ~kLeafBit) >> kLeafCountBits) - 1u;
        left = ref & kLeafMaxCount;
        g = gend = fl = 0u;
      } else {
        left = st >> kStMoreShift;
        g = gend = fl = 0u;
        if (st & kStGeometries) {
          const InstRec &in = p.insts[inst];
          g = geo + 1u;
          gend = in.geo_end;
          fl = merge_flags(r.flags, in.flags);
          F3 bd;
          stk.get_ray(o, bd);
          inv = recip(bd);
        }
      }
      for (;;) {
        if (g < gend) {
          const GeoRec &gr = p.geos[g];
          float tg;
          if (geometry_passes(fl, gr.flags) && slab(o, inv, near_, far_ * s, gr.mn[0], gr.mn[1], gr.mn[2], gr.mx[0],
                                                    gr.mx[1], gr.mx[2], tg)) {
            bool ce, cb;
            cull_triangle(fl, ce, cb);
            st = (st & (kStSecond | kStBack)) | (geometry_opaque(fl, gr.flags) ? kStOpaque : 0u) |
                 (ce ? kStCull : 0u) | (cb ? kStCullBack : 0u) | ((fl & F_END_SEARCH) ? kStEnd : 0u) |
                 (g + 1u < gend ? kStGeometries : 0u) | (left << kStMoreShift);
            geo = g;
            box = ray_box(o, inv);
            stk.push(kRefExit);  // the end mark of the BLAS, above the TLAS entries
            ref = LAYOUT ? gr.quad_root : gr.root_ref;
            break;
          }
          g++;
          continue;
        }
        if (left == 0u) {
          box = ray_box(r.o, winv);
          near_ = r.tmin;
          s = 1.0f;
          st |= kStWorld;
          ref = stk.pop();
          break;
        }
        inst++;
        left--;
        if constexpr (CNT) ci++;
        const InstRec &in = p.insts[inst];
        float ti;
        if (!slab(r.o, winv, r.tmin, far_, in.mn[0], in.mn[1], in.mn[2], in.mx[0], in.mx[1], in.mx[2], ti)) continue;
        if ((r.mask & in.mask) == 0u) continue;
        fl = merge_flags(r.flags, in.flags);
        if (fl & F_SKIP_TRIANGLES) continue;
        F3 bd;
        object_ray(in.inv, r.o, r.d, o, bd, s);
        stk.set_ray(o, bd);
        inv = recip(bd);
        near_ = r.tmin * s;
        g = in.geo_begin;
        gend = in.geo_end;
      }
    }
  }
}

// The register bound of a launch that asks for occupancy (TraceTune::waves):
// 96 registers, 5 waves per SIMD.  At 6 or 8 waves the kernels spill inside
// their loops (6 and 4 waves instead of 5: 1M rays in 100k triangles 3.4 and
// 4.7 % slower, a 1080p frame 5.8 and 7.1 %, an ambient-occlusion sample, whose
// launches are the cooperative kernel's, 10.5 and 4.9 %).
constexpr int kWavesBound = 5;

// Live slots of the first and the second segment of a launch.
__device__ __forceinline__ uint32_t live_first(const TraceParams &p) {
  return p.count ? min(slots_of(p), *p.count) : slots_of(p);
}
__device__ __forceinline__ uint32_t live_second(const TraceParams &p) {
  return p.count2 ? min(p.slots2, *p.count2) : 0u;
}
// The launch parameters of the second segment.
__device__ __forceinline__ void select_second(TraceParams &p) {
  p.rays = p.rays2;
  p.hits = p.hits2;
  p.hitx = p.hitx2;
  p.queue = p.queue2;
  p.flags = p.flags2;
  p.counters = nullptr;
}

// ------------------------------------------------------------------------
// Cooperative kernel: kCoopLanes consecutive lanes trace one ray.  Every lane
// of the group walks the TLAS in lockstep (same nodes, same far bound: the
// group's nearest hit so far); the instances it accepts are dealt to the
// lanes in batches of kCoopLanes, each lane walks its instance's BLAS alone,
// and after each batch the group takes the nearest far bound.  A ray's chain
// of dependent node loads becomes the TLAS walk plus the longest BLAS walk of
// each batch, which is what bounds small launches (the tail bounces of a
// path tracer): they last as long as their slowest ray.  The result is the
// nearest accepted hit, as in the one-ray-per-lane kernel; among hits with
// equal t the lowest lane of the last batch wins (a visit-order tie, as
// between the layouts).  Launches of at most kCoopWideMax rays give each ray
// 16 lanes: their time is their slowest rays' chains, and a batch of 16
// instances takes a ray over twice as many instances per BLAS round (the
// last bounces of the 1080p path-tracing frame: 2.88 -> 2.83 ms with every
// launch of at most 32k rays cooperative); larger launches keep 8, where
// the extra lanes cost more occupancy than they save.
// ------------------------------------------------------------------------
constexpr uint32_t kCoopLanes = 8;
constexpr uint32_t kCoopWideLanes = 16;
constexpr uint32_t kCoopWideMax = 32768;
// Inner steps go on while 1 / kCoopKeep of the wave's busy lanes want them
// (3 and 6 instead of 2: a 1080p frame 0.3 and 1.4 % slower, an
// ambient-occlusion sample 0.6 and 2.5 %).
constexpr uint32_t kCoopKeep = 2;

template <int G>
__device__ __forceinline__ float group_min(float v) {
  for (int m = G / 2; m > 0; m >>= 1) v = fminf(v, __shfl_xor(v, m, G));
  return v;
}
template <int G>
__device__ __forceinline__ bool group_any(bool b) {
  int v = b ? 1 : 0;
  for (int m = G / 2; m > 0; m >>= 1) v |= __shfl_xor(v, m, G);
  return v != 0;
}

// Returns (group-uniform) the lane of the group that wrote the record, plus
// kCoopHit when the ray hit.
constexpr uint32_t kCoopHit = 0x100u;

// The step of the lanes at an inner node.
template <int LAYOUT, class Stack>
__device__ __forceinline__ uint32_t inner_step(Stack &stk, const TraceParams &p, bool world, uint32_t ref,
                                               const RayBox &box, float tmin, float tmax) {
  if (LAYOUT == 0 || __ballot(!box.plain) == 0ull)  // wave-uniform
    return stk.template step<LAYOUT>([&]() { return test_kids<LAYOUT, true>(p, world, ref, box, tmin, tmax); });
  return stk.template step<LAYOUT>([&]() { return test_kids<LAYOUT, false>(p, world, ref, box, tmin, tmax); });
}

template <int K, int S, int B, int LAYOUT, int G = (int)kCoopLanes>
__device__ __forceinline__ uint32_t trace_coop_one(const TraceParams &p, uint32_t rid, uint32_t *lds,
                                                   uint32_t glane) {
  // the group's hit mask below is a 32-bit (1 << G) - 1
  static_assert(G == 8 || G == 16, "cooperative groups of 8 or 16 lanes");
  volatile uint32_t spill[LaneStack<K, S, B>::kSpill];
  LaneStack<K, S, B> stk{lds, spill, p.status, 0u};

  RayIn r = load_ray(p, rid);
  float far_ = r.tmax;  // group-uniform outside a batch's BLAS walks
  Best best;
  float best_t = 0.0f;  // this lane's own nearest accepted hit
  bool done = false;
  uint32_t cand = kInvalid, cnt = 0;

  // this lane's instance of the batch (already accepted by the TLAS walk);
  // as in trace_wave the lanes of the wave do one kind of work at a time
  auto run_instance = [&](uint32_t i) {
    const InstRec &in = p.insts[i];
    const uint32_t fl = merge_flags(r.flags, in.flags);
    float s;
    {
      F3 bo, bd;
      object_ray(in.inv, r.o, r.d, bo, bd, s);
      stk.set_ray(bo, bd);
    }
    const float near_s = r.tmin * s;
    uint32_t g = in.geo_begin, gend = in.geo_end, st = 0u, bref = kRefDone;
    RayBox box = {};
    // the first geometry from g on that the ray may hit
    auto enter = [&]() {
      F3 bo, bd;
      stk.get_ray(bo, bd);
      const F3 binv = recip(bd);
      bref = kRefDone;
      for (; g < gend; g++) {
        const GeoRec &geo = p.geos[g];
        float tg;
        if (!geometry_passes(fl, geo.flags) || !slab(bo, binv, near_s, far_ * s, geo.mn[0], geo.mn[1], geo.mn[2],
                                                     geo.mx[0], geo.mx[1], geo.mx[2], tg))
          continue;
        bool ce, cb;
        cull_triangle(fl, ce, cb);
        st = (geometry_opaque(fl, geo.flags) ? kStOpaque : 0u) | (ce ? kStCull : 0u) | (cb ? kStCullBack : 0u) |
             ((fl & F_END_SEARCH) ? kStEnd : 0u);
        box = ray_box(bo, binv);
        stk.push(kRefExit);  // above the TLAS entries
        bref = LAYOUT ? geo.quad_root : geo.root_ref;
        break;
      }
    };
    enter();
    for (;;) {
      const uint32_t a = wave_count(bref < kRefExit), b = wave_count((bref & kLeafBit) != 0u);
      if (a + b == 0u) break;
      if (a * kCoopKeep >= a + b) {
        if (bref < kRefExit) bref = inner_step<LAYOUT>(stk, p, false, bref, box, near_s, far_ * s);
      } else if (bref & kLeafBit) {
        const uint32_t k0 = (bref & ~kLeafBit) >> kLeafCountBits, k1 = k0 + (bref & kLeafMaxCount);
        F3 bo, bd;
        stk.get_ray(bo, bd);
        bref = stk.pop();
        for (uint32_t k = k0; k < k1; k++) {
          const float4 *q = reinterpret_cast<const float4 *>(p.tris + k);
          const float4 ta = q[0], tb = q[1], tc = q[2], td = q[3];
          float t, u, v;
          bool back;
          if (tri_core(bo, bd, near_s, far_ * s, f3(ta.x, ta.y, ta.z), f3(tb.x, tb.y, tb.z), f3(tc.x, tc.y, tc.z),
                       f3(td.x, td.y, td.z), ta.w, tb.w, tc.w, td.w, (st & kStCull) != 0u, (st & kStCullBack) != 0u, t,
                       u, v, back)) {
            uint32_t beh = (st & kStOpaque) ? RDRT_ANYHIT_ACCEPT : anyhit_behavior(p, false, p.tri_ids[k]);
            if (beh & RDRT_ANYHIT_ACCEPT) {
              far_ = t / s;
              best_t = far_;
              best.k = k;
              best.geo = g;
              best.inst = i;
              best.u = u;
              best.v = v;
              best.back = back;
              if (st & kStEnd) beh |= RDRT_ANYHIT_END_SEARCH;
            }
            if (beh & RDRT_ANYHIT_END_SEARCH) {
              done = true;
              bref = kRefDone;
              break;
            }
          }
        }
      }
      if (bref == kRefExit) {
        g++;
        if (g < gend) enter();
        else bref = kRefDone;
      }
    }
  };
  // every lane of the group: walk the batch, then share the far bound
  auto flush = [&]() {
    if (cand != kInvalid) run_instance(cand);
    cand = kInvalid;
    cnt = 0;
    far_ = group_min<G>(far_);
    done = group_any<G>(done);
    r = load_ray(p, rid);
  };

  const TlasRoot *root = bound_root(p, r.tlas_idx);
  F3 winv = recip(r.d);
  float tn;
  if (root && slab(r.o, winv, r.tmin, far_, root->mn[0], root->mn[1], root->mn[2], root->mx[0], root->mx[1],
                   root->mx[2], tn)) {
    uint32_t ref = LAYOUT ? p.tlas_quad_roots[root - p.tlas_roots] : root->root_ref;
    stk.push(kRefDone);
    RayBox box = ray_box(r.o, winv);
    while (ref != kRefDone) {
      if (!(ref & kLeafBit)) {
        ref = inner_step<LAYOUT>(stk, p, true, ref, box, r.tmin, far_);
      } else {
        const uint32_t i0 = (ref & ~kLeafBit) >> kLeafCountBits, i1 = i0 + (ref & kLeafMaxCount);
        for (uint32_t i = i0; i < i1 && !done; i++) {
          const InstRec &in = p.insts[i];
          float ti;
          if (!slab(r.o, winv, r.tmin, far_, in.mn[0], in.mn[1], in.mn[2], in.mx[0], in.mx[1], in.mx[2], ti))
            continue;
          if ((r.mask & in.mask) == 0) continue;
          if (merge_flags(r.flags, in.flags) & F_SKIP_TRIANGLES) continue;
          if (glane == cnt) cand = i;
          if (++cnt == (uint32_t)G) {
            flush();
            winv = recip(r.d);
            box = ray_box(r.o, winv);
          }
        }
        if (done) break;
        ref = stk.pop();
      }
    }
    if (cnt) flush();
  }
  // the lowest lane whose own hit is the group's nearest reports it
  const bool mine = best.k != kInvalid && best_t == far_;
  const uint64_t m = __ballot(mine);
  const uint32_t lane = __lane_id();
  const uint32_t gm = (uint32_t)(m >> (lane & ~((uint32_t)G - 1u))) & ((1u << G) - 1u);
  const uint32_t win = gm ? (uint32_t)__ffs(gm) - 1u : 0u;
  if (glane == win) {
    if (!gm) best.k = kInvalid;
    best.t = far_;
    write_result(p, p.tri_ids, rid, best, 0u, 0u, 0u);
  }
  return win | (gm ? kCoopHit : 0u);
}

// G lanes per ray: group gi of the grid takes the gi-th live ray.
template <int K, int S, int B, int LAYOUT, int G>
__device__ __forceinline__ void trace_coop_group(TraceParams &p, uint32_t n0, uint32_t n1, uint32_t *lds) {
  const uint32_t gi = (blockIdx.x * B + threadIdx.x) / (uint32_t)G;
  uint32_t slot = gi, n = n0;
  if (gi >= n0) {
    slot = gi - n0;
    n = n1;
    select_second(p);
  }
  if (slot >= n) return;  // whole groups: the lanes of a group share gi
  const uint32_t rid = p.queue ? p.queue[slot] : slot;
  if (rid >= p.n) return;
  trace_coop_one<K, S, B, LAYOUT, G>(p, rid, lds + threadIdx.x, threadIdx.x & ((uint32_t)G - 1u));
}

template <int K, int S, int B, int LAYOUT>
__global__ __launch_bounds__(B, kWavesBound) void k_trace_coop(TraceParams p) {
  __shared__ uint32_t lds[LaneStack<K, S, B>::kRows * B];
  const uint32_t n0 = live_first(p), n1 = live_second(p);
  if (n0 + n1 > p.coop_max) return;  // the one-ray-per-lane kernel traces launches this large
  // the group width is uniform over the launch (the live count is)
  if (n0 + n1 <= kCoopWideMax) trace_coop_group<K, S, B, LAYOUT, (int)kCoopWideLanes>(p, n0, n1, lds);
  else trace_coop_group<K, S, B, LAYOUT, (int)kCoopLanes>(p, n0, n1, lds);
}

// Rays that a wave starts with.  A launch that leaves SIMDs idle lasts as long
// as its slowest wave, and a wave takes the steps of all its rays, so few rays
// go to each, until there are two waves per SIMD (4096 rays in 2000 triangles:
// 59.6 us in 64 waves of 64, 47.0 in 512 of 8; 21k paths in 64 meshes: 477 and
// 419 us; 1024 or 4096 waves are within 4 % of 2048).
constexpr uint32_t kSpreadWaves = 2048, kFewestRays = 8;
__host__ __device__ inline uint32_t rays_per_wave(uint32_t total, uint32_t waves) {
  uint32_t r = kFewestRays;
  const uint32_t w = waves < kSpreadWaves ? waves : kSpreadWaves;
  while (r < 64u && (total + r - 1u) / r > w) r *= 2u;
  return r;
}

// One ray per thread, or fewer rays than lanes in a small launch, over a grid
// sized for both segments' slots; the live counts may be smaller (device queue
// sizes).
template <int K, int S, int B, int W, bool CNT, int LAYOUT>
__global__ __launch_bounds__(B, W) void k_trace_fast(TraceParams p) {
  __shared__ uint32_t lds[LaneStack<K, S, B>::kRows * B];
  const uint32_t n0 = live_first(p), n1 = live_second(p);
  if (p.coop_max && n0 + n1 <= p.coop_max) return;  // the cooperative kernel traces it
  const uint32_t total = n0 + n1, per = rays_per_wave(total, gridDim.x * (B / 64u)), block = per * (B / 64u);
  const uint32_t used = (total + block - 1u) / block;
  if (blockIdx.x >= used) return;
  const uint32_t first = xcd_block(blockIdx.x, used) * block + (threadIdx.x >> 6) * per;
  if (first >= total) return;  // whole waves
  trace_wave<K, S, B, CNT, LAYOUT>(p, n0, __builtin_amdgcn_readfirstlane(first),
                                   __builtin_amdgcn_readfirstlane(min(total, first + per)), lds + threadIdx.x,
                                   [](uint32_t &, uint32_t &) { return false; });
}

// Persistent variant: a grid sized to the resident capacity whose waves pull
// chunks of consecutive queue slots until the queue is exhausted, so uneven
// rays and scenes balance across the chip.  The slots are divided among the
// XCDs (blocks are dispatched to them round-robin), so that neighbouring rays
// share an L2; a wave whose XCD's share is exhausted helps the next one.
// Every share has a counter of its own: atomics on one address come out one
// every ~18 ns, which on a single counter held a launch of 2M rays in chunks
// of 64 at 0.7 ms whatever the rays took.  A wave's first chunk is the one of
// its index, without an atomic; an empty launch, or one whose shares those
// chunks cover, has none at all (with them, eight for every wave, an empty
// launch took 64 us longer than the plain kernel's, 1.6 us now; a 1080p pipeline
// call, most of whose launches are empty, 1.87 -> 1.49 ms).  Reading a share's
// counter before adding to it, so that waves leave exhausted shares alone,
// made filled launches slower (2M camera rays: 567 -> 645 us).  Every wave
// exits once each share is drained.
template <int K, int S, int B, int W, bool CNT, int LAYOUT>
__global__ __launch_bounds__(B, W) void k_trace_persist(TraceParams p) {
  __shared__ uint32_t lds[LaneStack<K, S, B>::kRows * B];
  const uint32_t n0 = live_first(p), n1 = live_second(p);
  if (p.coop_max && n0 + n1 <= p.coop_max) return;  // the cooperative kernel traces it
  const uint32_t total = n0 + n1;
  if (total == 0u) return;
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr uint32_t kWaves = B / 64u;
  const uint32_t share = (total / kWorkGroups + 63u) & ~63u;  // slots of one XCD, in whole chunks
  // chunks of 64, larger when a wave has very many to pull (5M rays in 2000
  // triangles: 390 us in chunks of 64, 358 of 128; 16M: 1170 and 1106), smaller
  // when the first ones already leave waves without rays
  const uint32_t chunk = total >= (1u << 22) ? 128u : rays_per_wave(total, gridDim.x * kWaves);
  uint32_t tried = 0;      // shares found drained
  bool own = true;         // the first chunk is not taken yet
  trace_wave<K, S, B, CNT, LAYOUT>(p, n0, 0u, 0u, lds + threadIdx.x, [&](uint32_t &next, uint32_t &end) {
    while (tried < kWorkGroups) {
      const uint32_t g = (blockIdx.x + tried) % kWorkGroups;
      const uint32_t first = g * share, stop = g + 1u == kWorkGroups ? total : min(total, first + share);
      // the chunks of the group's own waves come first
      const uint32_t waves = (gridDim.x - g + kWorkGroups - 1u) / kWorkGroups * kWaves;
      uint32_t at;
      if (own) {
        own = false;
        at = (blockIdx.x / kWorkGroups * kWaves + wave) * chunk;
      } else {
        if (first + waves * chunk >= stop) {  // nothing behind the first chunks
          tried++;
          continue;
        }
        uint32_t add = 0;
        if (lane == 0) add = atomicAdd(p.work + g * kWorkStride, chunk);
        at = waves * chunk + __builtin_amdgcn_readfirstlane(add);
      }
      if (first < stop && at < stop - first) {
        next = first + at;
        end = min(stop, next + chunk);
        return true;
      }
      tried++;
    }
    return false;
  });
}

// Blocks of a launch: a lane for every slot, or a wave for every kFewestRays
// slots of a launch too small for kSpreadWaves waves of 64.
inline uint32_t spread_grid(const TraceParams &p, uint32_t block) {
  const uint32_t blocks = grid_slots(p, block) / block, most = (kSpreadWaves * 64u + block - 1u) / block;
  return blocks >= most ? blocks : std::min(most, blocks * (64u / kFewestRays));
}

[[maybe_unused]] __global__ void k_zero_work(uint32_t *w) { clear_work(w, threadIdx.x); }

// One fast-traversal launch with block size B, total stack S and tuning t.
// K = stack entries per lane in LDS, W = minimum waves per SIMD asked of the
// register allocator (1 = its own choice), LAYOUT = TraceTune::wide.
template <int K, int S, int B, int W, int LAYOUT>
hipError_t launch_fast_kw(const TraceParams &p0, bool persist, uint32_t coop, hipStream_t st) {
  TraceParams p = p0;
  p.coop_max = p.counters ? 0u : coop;  // visit counting stays one ray per lane
  if (p.coop_max) {
    // enough groups for every live ray when the launch qualifies
    uint32_t live = slots_of(p) + (p.count2 ? p.slots2 : 0u);
    if (p.live_max && p.live_max < live) live = p.live_max;
    const uint32_t groups = std::min(p.coop_max, live);
    // 8 lanes per ray, or 16 when at most kCoopWideMax rays are live
    const uint32_t threads = std::max(groups * kCoopLanes, std::min(groups, kCoopWideMax) * kCoopWideLanes);
    const uint32_t grid = (threads + B - 1) / B;
    if (grid) hipLaunchKernelGGL((k_trace_coop<K, S, B, LAYOUT>), dim3(grid), dim3(B), 0, st, p);
    if (live <= p.coop_max) return hipGetLastError();  // the cooperative kernel always qualifies
  }
  if (persist) {
    if (!p.work) return hipErrorInvalidValue;
    if (!p.work_zeroed) hipLaunchKernelGGL(k_zero_work, dim3(1), dim3(64), 0, st, p.work);
    if (p.counters) {
      auto k = k_trace_persist<K, S, B, W, true, LAYOUT>;
      uint32_t g = std::min(resident_grid((const void *)k, B), spread_grid(p, B));
      hipLaunchKernelGGL(k, dim3(g), dim3(B), 0, st, p);
    } else {
      auto k = k_trace_persist<K, S, B, W, false, LAYOUT>;
      uint32_t g = std::min(resident_grid((const void *)k, B), spread_grid(p, B));
      hipLaunchKernelGGL(k, dim3(g), dim3(B), 0, st, p);
    }
    return hipGetLastError();
  }
  dim3 grid(spread_grid(p, B));
  if (p.counters) hipLaunchKernelGGL((k_trace_fast<K, S, B, W, true, LAYOUT>), grid, dim3(B), 0, st, p);
  else hipLaunchKernelGGL((k_trace_fast<K, S, B, W, false, LAYOUT>), grid, dim3(B), 0, st, p);
  return hipGetLastError();
}

template <int S, int B, int LAYOUT>
hipError_t launch_fast_s(const TraceParams &p, const TraceTune &t, hipStream_t st) {
  constexpr int K8 = S < 8 ? S : 8;
  constexpr int K16 = S < 16 ? S : 16;
  const bool persist = t.persist != 0;
  if (t.waves) {
    if (t.lds <= 8) return launch_fast_kw<K8, S, B, kWavesBound, LAYOUT>(p, persist, t.coop, st);
    return launch_fast_kw<K16, S, B, kWavesBound, LAYOUT>(p, persist, t.coop, st);
  }
  if (t.lds <= 8) return launch_fast_kw<K8, S, B, 1, LAYOUT>(p, persist, t.coop, st);
  return launch_fast_kw<K16, S, B, 1, LAYOUT>(p, persist, t.coop, st);
}

template <int B, int LAYOUT>
hipError_t launch_fast_block(const TraceParams &p, uint32_t s, const TraceTune &t, hipStream_t st) {
  switch (s) {
    case 8: return launch_fast_s<8, B, LAYOUT>(p, t, st);
    case 16: return launch_fast_s<16, B, LAYOUT>(p, t, st);
    case 24: return launch_fast_s<24, B, LAYOUT>(p, t, st);
    case 32: return launch_fast_s<32, B, LAYOUT>(p, t, st);
    case 48: return launch_fast_s<48, B, LAYOUT>(p, t, st);
    case 64: return launch_fast_s<64, B, LAYOUT>(p, t, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace
}  // namespace rdrt

#endif
