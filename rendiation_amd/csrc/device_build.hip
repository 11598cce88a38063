// device_build.hip -- BLAS trees built on the device, level by level.
//
// Both trees of a geometry are built with the host builders' semantics
// (bvh_build.cpp), so they are node for node the same trees:
//  * the reference's tree: binned SAH on the longest axis of the node box,
//    nb <= 4 bins, first strict minimum of area(L)|L| + area(R)|R|, a stable
//    reorder by bin, the median split when every centre lands in one bin
//    (strategy.rs:99-285; the order inside each half follows a stable sort
//    by centre, where the host follows std::nth_element: only the order
//    inside leaves after a median split can differ);
//  * the fast kernels' tree: 16 bins on each axis of the centre bounds, SAH
//    in FP64 with a leaf when cheaper (at most max_leaf primitives), a stable
//    two-way partition, the object median when every centre coincides.
//
// One level is a handful of launches over all primitives (centre bounds,
// binning with block-private LDS bins when a block lies in one node, a
// node-parallel split, the partition keys, a scan and a scatter).  Node
// bounds and bin boxes are unions, exact in any order (float min / max as
// ordered-integer atomics), and the split arithmetic is the host's operation
// for operation, so the decisions are the host's.  The host converts the
// level-order nodes to the preorder Tree.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "device_build.h"

#pragma clang fp contract(off)

namespace rdrt {
namespace {

// f(i) for i < n on the host's threads (each index once).
template <class F>
void host_for(size_t n, F f) {
  const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
  const unsigned threads = (unsigned)std::min<size_t>(hw, n);
  if (threads <= 1) {
    for (size_t i = 0; i < n; i++) f(i);
    return;
  }
  std::atomic<size_t> next{0};
  std::vector<std::thread> pool;
  for (unsigned w = 0; w < threads; w++)
    pool.emplace_back([&] {
      for (size_t i; (i = next.fetch_add(1)) < n;) f(i);
    });
  for (auto &th : pool) th.join();
}

constexpr uint32_t kB = 256;          // threads per block
constexpr uint32_t kFastBins = 16;    // FastTreeOptions::bins the device supports
constexpr uint32_t kMaxRefBins = 4;   // reference bins the device supports
constexpr uint32_t kMaxSlotWords = 3 * kFastBins * 7;

using u32 = uint32_t;

// ordered-integer keys of floats: u < v <=> f(u) < f(v) (finite or infinite)
__device__ __forceinline__ u32 fkey(float f) {
  const u32 u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float funkey(u32 k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
constexpr u32 kMinInit = 0xffffffffu;  // identity of a min over keys
constexpr u32 kMaxInit = 0u;           // identity of a max over keys

struct DBox {
  float mn[3], mx[3];
};
__device__ __forceinline__ DBox dempty() {
  const float inf = __builtin_inff();
  return DBox{{inf, inf, inf}, {-inf, -inf, -inf}};
}
__device__ __forceinline__ void dgrow(DBox &b, const DBox &o) {
  for (int k = 0; k < 3; k++) {
    b.mn[k] = fminf(b.mn[k], o.mn[k]);
    b.mx[k] = fmaxf(b.mx[k], o.mx[k]);
  }
}
// box3.rs:5-11
__device__ __forceinline__ float darea(const DBox &b) {
  const float w = b.mx[0] - b.mn[0], h = b.mx[1] - b.mn[1], d = b.mx[2] - b.mn[2];
  return 2.0f * (w * h + w * d + h * d);
}
// box3.rs:117-133
__device__ __forceinline__ int dlongest(const DBox &b) {
  const float x = b.mx[0] - b.mn[0], y = b.mx[1] - b.mn[1], z = b.mx[2] - b.mn[2];
  if (x > y) return x > z ? 0 : 2;
  return y > z ? 1 : 2;
}

// The builder's device state for one geometry of n primitives.
struct Dev {
  u32 n;
  const float *pbox;   // 6 per primitive
  float *cen;          // 3 per primitive
  u32 *order, *order2, *node_of, *node_of2;
  uint4 *keys;         // one-hot partition key per position (n + 1)
  uint4 *scan;         // exclusive scan of keys (n + 1)
  uint4 *bsum;         // scan block sums
  // nodes
  float *nbox;         // 6 per node
  u32 *nbeg, *nend, *ndepth, *nchild, *nflags;  // flags: 1 inner, 2 median split
  u32 *nlc;            // reference: left count of a split (its split point is begin + lc)
  int *naxis;
  float *na, *ns;      // bin origin and step (reference) or centre min and scale (fast)
  u32 *nbest;          // fast: best bin
  u32 *nright, *ngeo;  // right-child steps on the path from the root; geometry
  u32 *count;          // [0] node count, [1] median splits this level, [2] error bits, [3] next level's begin
  u32 cap;             // node capacity
  // per active slot
  u32 *cb;             // 6 keys per slot (centre bounds, fast)
  u32 *bins;           // kMaxSlotWords per slot: counts then box keys
  u32 lo, m;           // active nodes [lo, lo + m)
  u32 mode;            // 0 reference, 1 fast
  u32 K, axes;         // bins per axis, binned axes
  u32 max_depth, bin_size, max_leaf;
  double node_cost, prim_cost;
};

__device__ __forceinline__ DBox prim_box(const Dev &d, u32 p) {
  const float *q = d.pbox + 6 * (size_t)p;
  return DBox{{q[0], q[1], q[2]}, {q[3], q[4], q[5]}};
}
constexpr u32 kDone = 8u;    // node flag: its subtree was built whole by one wave (k_small)
constexpr u32 kSmall = 64u;  // nodes of at most this many primitives are built by one wave

// A node of this level still built by the level kernels.
__device__ __forceinline__ bool active(const Dev &d, u32 nd) {
  return nd != kInvalid && nd - d.lo < d.m && !(d.nflags[nd] & kDone);
}

// One block's primitives all lie in one node when its first and last do
// (node ranges are contiguous).  Returns that node or kInvalid.
__device__ u32 block_node(const Dev &d) {
  __shared__ u32 s_nd;
  if (threadIdx.x == 0) {
    const u32 first = blockIdx.x * kB, last = min(first + kB, d.n) - 1;
    const u32 a = d.node_of[first], b = d.node_of[last];
    s_nd = (a == b && active(d, a)) ? a : kInvalid;
  }
  __syncthreads();
  return s_nd;
}

// Centres, the identity order and every primitive's root (geometry g's
// root is node g; geo_of holds it per primitive).
__global__ __launch_bounds__(kB) void k_centres(Dev d, const u32 *geo_of) {
  const u32 i = blockIdx.x * kB + threadIdx.x;
  if (i >= d.n) return;
  const DBox b = prim_box(d, i);
  for (int k = 0; k < 3; k++) d.cen[3 * (size_t)i + k] = (b.mn[k] + b.mx[k]) * 0.5f;  // box3.rs:90-93
  d.order[i] = i;
  d.node_of[i] = geo_of[i];
}

// Folds the lanes' keys c (3 minima, 3 maxima) into keys[6 * slot]: a wave
// meets few nodes, whose ranges are contiguous, so each node's lanes are
// reduced in registers and 6 lanes add the result.  An atomic per lane and key
// made k_centre_bounds 100 us on a level of 100k triangles (LDS words where a
// block had one node); 7 us now.  Whole waves call this (slot kInvalid:
// nothing to add).
__device__ __forceinline__ void fold_keys(u32 *keys, u32 slot, const u32 c[6]) {
  const u32 lane = threadIdx.x & 63u;
  unsigned long long todo = __ballot(slot != kInvalid);
  while (todo) {
    const u32 of = (u32)__shfl((int)slot, __ffsll(todo) - 1, 64);
    const bool mine = slot == of;
    todo &= ~__ballot(mine);
    u32 out = 0;
    for (u32 k = 0; k < 6; k++) {
      u32 v = mine ? c[k] : k < 3 ? kMinInit : kMaxInit;
      for (int o = 32; o > 0; o >>= 1) {
        const u32 w = (u32)__shfl_xor((int)v, o, 64);
        v = k < 3 ? min(v, w) : max(v, w);
      }
      if (lane == k) out = v;
    }
    if (lane < 3) atomicMin(&keys[6 * (size_t)of + lane], out);
    else if (lane < 6) atomicMax(&keys[6 * (size_t)of + lane], out);
  }
}

// Union of the primitive boxes of every active node flagged `want` (1 =
// all, 2 = children of median splits, whose boxes are range unions), into
// nbox as keys first (nbox reinterpreted), decoded by k_decode_boxes.
__global__ __launch_bounds__(kB) void k_range_boxes(Dev d, u32 *keys) {
  __shared__ u32 s[6];
  const u32 nd_block = block_node(d);
  if (nd_block != kInvalid && threadIdx.x < 6) s[threadIdx.x] = threadIdx.x < 3 ? kMinInit : kMaxInit;
  __syncthreads();
  const u32 i = blockIdx.x * kB + threadIdx.x;
  u32 slot = kInvalid, c[6] = {};
  if (i < d.n) {
    const u32 nd = d.node_of[i];
    if (active(d, nd)) {
      const DBox b = prim_box(d, d.order[i]);
      slot = nd_block != kInvalid ? 0u : nd - d.lo;
      for (int k = 0; k < 3; k++) {
        c[k] = fkey(b.mn[k]);
        c[3 + k] = fkey(b.mx[k]);
      }
    }
  }
  fold_keys(nd_block != kInvalid ? s : keys, slot, c);
  __syncthreads();
  if (nd_block != kInvalid && threadIdx.x < 6) {
    u32 *q = keys + 6 * (size_t)(nd_block - d.lo);
    if (threadIdx.x < 3) atomicMin(&q[threadIdx.x], s[threadIdx.x]);
    else atomicMax(&q[threadIdx.x], s[threadIdx.x]);
  }
}

__global__ void k_decode_boxes(Dev d, const u32 *keys, u32 want) {
  const u32 j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= d.m) return;
  const u32 nd = d.lo + j;
  if (want == 2 && !(d.nflags[nd] & 4u)) return;  // only children of median splits
  const bool empty = d.nbeg[nd] == d.nend[nd];     // a geometry without triangles
  for (int k = 0; k < 6; k++)
    d.nbox[6 * (size_t)nd + k] = empty ? (k < 3 ? __builtin_inff() : -__builtin_inff()) : funkey(keys[6 * (size_t)j + k]);
}

// Centre bounds of every active node (fast tree).
__global__ __launch_bounds__(kB) void k_centre_bounds(Dev d) {
  __shared__ u32 s[6];
  const u32 nd_block = block_node(d);
  if (nd_block != kInvalid && threadIdx.x < 6) s[threadIdx.x] = threadIdx.x < 3 ? kMinInit : kMaxInit;
  __syncthreads();
  const u32 i = blockIdx.x * kB + threadIdx.x;
  u32 slot = kInvalid, c[6] = {};
  if (i < d.n) {
    const u32 nd = d.node_of[i];
    if (active(d, nd)) {
      const u32 p = d.order[i];
      slot = nd_block != kInvalid ? 0u : nd - d.lo;
      for (int k = 0; k < 3; k++) c[k] = c[3 + k] = fkey(d.cen[3 * (size_t)p + k]);
    }
  }
  fold_keys(nd_block != kInvalid ? s : d.cb, slot, c);
  __syncthreads();
  if (nd_block != kInvalid && threadIdx.x < 6) {
    u32 *q = d.cb + 6 * (size_t)(nd_block - d.lo);
    if (threadIdx.x < 3) atomicMin(&q[threadIdx.x], s[threadIdx.x]);
    else atomicMax(&q[threadIdx.x], s[threadIdx.x]);
  }
}

// Per active node: the binning parameters.  Reference: the longest axis of
// the node box, origin and step of nb bins; fast: per axis the centre
// minimum and K / extent (0 when the axis is not live).
__global__ void k_prep(Dev d) {
  const u32 j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= d.m) return;
  if (j == 0) d.count[3] = d.count[0];  // k_small's nodes end here: the next level begins
  const u32 nd = d.lo + j;
  if (d.nflags[nd] & kDone) return;
  if (d.mode == 0) {
    DBox b;
    for (int k = 0; k < 3; k++) {
      b.mn[k] = d.nbox[6 * (size_t)nd + k];
      b.mx[k] = d.nbox[6 * (size_t)nd + 3 + k];
    }
    const int axis = dlongest(b);
    d.naxis[nd] = axis;
    d.na[3 * (size_t)nd] = b.mn[axis];
    d.ns[3 * (size_t)nd] = (b.mx[axis] - b.mn[axis]) / (float)d.K;
  } else {
    for (int k = 0; k < 3; k++) {
      const float cmn = funkey(d.cb[6 * (size_t)j + k]), cmx = funkey(d.cb[6 * (size_t)j + 3 + k]);
      const float ext = cmx - cmn;
      d.na[3 * (size_t)nd + k] = cmn;
      d.ns[3 * (size_t)nd + k] = ext > 0.0f ? (float)d.K / ext : 0.0f;
    }
  }
}

// Bin of a centre: the host's formulas (bvh_build.cpp sah_split / bin_of).
__device__ __forceinline__ u32 ref_bin(float c, float a0, float step, u32 nb) {
  const float f = floorf((c - a0) / step);
  size_t w = 0;
  if (f > 0.0f) w = f >= 1.8446744e19f ? ~(size_t)0 : (size_t)f;  // Rust's saturating cast
  if (w >= nb) w = nb - 1;
  return (u32)w;
}
__device__ __forceinline__ u32 fast_bin(float c, float mn, float scale, u32 K) {
  return (u32)fminf((float)(K - 1), fmaxf(0.0f, (c - mn) * scale));
}

// Bin counts and boxes of every active node; slot layout: counts[axes * K],
// then box keys [axes * K][6].
__global__ __launch_bounds__(kB) void k_bins(Dev d) {
  __shared__ u32 s[kMaxSlotWords];
  const u32 words = d.axes * d.K * 7;
  const u32 nd_block = block_node(d);
  if (nd_block != kInvalid)
    for (u32 w = threadIdx.x; w < words; w += kB) {
      const u32 box = w - d.axes * d.K;
      s[w] = w < d.axes * d.K ? 0u : ((box % 6) < 3 ? kMinInit : kMaxInit);
    }
  __syncthreads();
  const u32 i = blockIdx.x * kB + threadIdx.x;
  if (i < d.n) {
    const u32 nd = d.node_of[i];
    if (active(d, nd)) {
      const u32 p = d.order[i];
      const DBox b = prim_box(d, p);
      u32 *q = nd_block != kInvalid ? s : d.bins + (size_t)kMaxSlotWords * (nd - d.lo);
      for (u32 a = 0; a < d.axes; a++) {
        u32 w;
        if (d.mode == 0) {
          const int axis = d.naxis[nd];
          w = ref_bin(d.cen[3 * (size_t)p + axis], d.na[3 * (size_t)nd], d.ns[3 * (size_t)nd], d.K);
        } else {
          const float sc = d.ns[3 * (size_t)nd + a];
          if (!(sc > 0.0f)) continue;  // axis not live
          w = fast_bin(d.cen[3 * (size_t)p + a], d.na[3 * (size_t)nd + a], sc, d.K);
        }
        const u32 slot = a * d.K + w;
        atomicAdd(&q[slot], 1u);
        u32 *bk = q + d.axes * d.K + 6 * slot;
        for (int k = 0; k < 3; k++) {
          atomicMin(&bk[k], fkey(b.mn[k]));
          atomicMax(&bk[3 + k], fkey(b.mx[k]));
        }
      }
    }
  }
  __syncthreads();
  if (nd_block != kInvalid) {
    u32 *q = d.bins + (size_t)kMaxSlotWords * (nd_block - d.lo);
    for (u32 w = threadIdx.x; w < words; w += kB) {
      if (w < d.axes * d.K) {
        if (s[w]) atomicAdd(&q[w], s[w]);
      } else if (((w - d.axes * d.K) % 6) < 3) {
        if (s[w] != kMinInit) atomicMin(&q[w], s[w]);
      } else if (s[w] != kMaxInit) {
        atomicMax(&q[w], s[w]);
      }
    }
  }
}

__device__ __forceinline__ DBox bin_box(const Dev &d, const u32 *q, u32 slot) {
  if (q[slot] == 0) return dempty();
  const u32 *bk = q + d.axes * d.K + 6 * slot;
  return DBox{{funkey(bk[0]), funkey(bk[1]), funkey(bk[2])}, {funkey(bk[3]), funkey(bk[4]), funkey(bk[5])}};
}

constexpr u32 kErrNodes = 1u, kErrMedian = 2u;
constexpr u32 kMaxMedianSort = 4096;  // primitives of a reference median split sorted by one thread

__device__ void new_children(Dev &d, u32 nd, const DBox &lb, const DBox &rb, u32 mid, bool median) {
  const u32 c = atomicAdd(&d.count[0], 2u);
  if (c + 2u > d.cap) {  // only with degenerate options (bin_size 0): reported, nothing written
    atomicOr(&d.count[2], kErrNodes);
    return;
  }
  if (median && d.mode == 0 && d.nend[nd] - d.nbeg[nd] > kMaxMedianSort) {
    atomicOr(&d.count[2], kErrMedian);
    return;
  }
  const u32 b = d.nbeg[nd], e = d.nend[nd], depth = d.ndepth[nd] + 1;
  const DBox kids[2] = {lb, rb};
  const u32 beg[2] = {b, mid}, end[2] = {mid, e};
  for (int s = 0; s < 2; s++) {
    for (int k = 0; k < 3; k++) {
      d.nbox[6 * (size_t)(c + s) + k] = kids[s].mn[k];
      d.nbox[6 * (size_t)(c + s) + 3 + k] = kids[s].mx[k];
    }
    d.nbeg[c + s] = beg[s];
    d.nend[c + s] = end[s];
    d.ndepth[c + s] = depth;
    d.nchild[c + s] = kInvalid;
    d.nflags[c + s] = median ? 4u : 0u;
    d.nright[c + s] = d.nright[nd] + (u32)s;
    d.ngeo[c + s] = d.ngeo[nd];
  }
  d.nchild[nd] = c;
  d.nflags[nd] |= 1u | (median ? 2u : 0u);
  d.nlc[nd] = mid - b;
  if (median) atomicAdd(&d.count[1], 1u);
}

// Split decision of every active node (one thread per node).
__global__ void k_split(Dev d) {
  const u32 j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= d.m) return;
  const u32 nd = d.lo + j;
  if (d.nflags[nd] & kDone) return;
  const u32 b = d.nbeg[nd], e = d.nend[nd], n = e - b, depth = d.ndepth[nd];
  const u32 *q = d.bins + (size_t)kMaxSlotWords * j;
  DBox nb;
  for (int k = 0; k < 3; k++) {
    nb.mn[k] = d.nbox[6 * (size_t)nd + k];
    nb.mx[k] = d.nbox[6 * (size_t)nd + 3 + k];
  }
  d.nchild[nd] = kInvalid;
  if (d.mode == 0) {
    if (!(depth < d.max_depth && n > d.bin_size)) return;  // utils.rs:20-37
    const u32 K = d.K;
    u32 empty = 0;
    for (u32 k = 0; k < K; k++) empty += q[k] == 0 ? 1u : 0u;
    if (empty == K - 1) {
      new_children(d, nd, dempty(), dempty(), b + n / 2, true);  // median: boxes after the sort
      return;
    }
    float best_cost = __builtin_inff();
    DBox best_l = dempty(), best_r = dempty();
    u32 best_lc = 0;
    for (u32 s = 0; s + 1 < K; s++) {
      DBox l = dempty(), r = dempty();
      u32 lc = 0, rc = 0;
      for (u32 k = 0; k <= s; k++) {
        lc += q[k];
        dgrow(l, bin_box(d, q, k));
      }
      for (u32 k = s + 1; k < K; k++) {
        rc += q[k];
        dgrow(r, bin_box(d, q, k));
      }
      const float cost = darea(l) * (float)lc + darea(r) * (float)rc;
      if (cost < best_cost) {
        best_cost = cost;
        best_l = l;
        best_r = r;
        best_lc = lc;
      }
    }
    new_children(d, nd, best_l, best_r, b + best_lc, false);
    return;
  }
  // fast tree
  if (n <= 1 || depth >= d.max_depth) return;
  bool any = false;
  for (int k = 0; k < 3; k++) any |= d.ns[3 * (size_t)nd + k] > 0.0f;
  if (!any) {
    new_children(d, nd, dempty(), dempty(), b + n / 2, true);  // object median: boxes from the ranges
    return;
  }
  const u32 K = d.K;
  const float parent_area = darea(nb);
  double best_cost = __builtin_inf();
  int best_axis = -1;
  u32 best_bin = 0;
  double right_cost[kFastBins];
  for (int axis = 0; axis < 3; axis++) {
    if (!(d.ns[3 * (size_t)nd + axis] > 0.0f)) continue;
    const u32 *c = q + axis * K;
    DBox r = dempty();
    u32 rc = 0;
    for (u32 k = K - 1; k >= 1; k--) {
      dgrow(r, bin_box(d, q, axis * K + k));
      rc += c[k];
      right_cost[k] = (double)darea(r) * rc;
    }
    DBox l = dempty();
    u32 lc = 0;
    for (u32 k = 0; k + 1 < K; k++) {
      dgrow(l, bin_box(d, q, axis * K + k));
      lc += c[k];
      if (lc == 0 || lc == n) continue;
      const double cost = (double)darea(l) * lc + right_cost[k + 1];
      if (cost < best_cost) {
        best_cost = cost;
        best_axis = axis;
        best_bin = k;
      }
    }
  }
  const double split_cost = d.node_cost + d.prim_cost * best_cost / fmax((double)parent_area, 1e-30);
  if (n <= d.max_leaf && split_cost >= d.prim_cost * n) return;  // leaf
  if (best_axis < 0) return;  // unreachable: a live axis always has a split
  DBox lb = dempty(), rb = dempty();
  u32 lc = 0;
  for (u32 k = 0; k < K; k++) {
    dgrow(k <= best_bin ? lb : rb, bin_box(d, q, best_axis * K + k));
    if (k <= best_bin) lc += q[best_axis * K + k];
  }
  d.naxis[nd] = best_axis;
  d.nbest[nd] = best_bin;
  new_children(d, nd, lb, rb, b + lc, false);
}

// Reference median split: sorts the node's range by centre on the longest
// axis (stable: ties keep their order).  One thread per node; these nodes
// are rare (every centre in one bin).
__global__ void k_median_sort(Dev d) {
  const u32 j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= d.m) return;
  const u32 nd = d.lo + j;
  if (d.nflags[nd] & kDone) return;
  if (!(d.nflags[nd] & 2u) || d.mode != 0) return;
  const u32 b = d.nbeg[nd], e = d.nend[nd];
  const int axis = d.naxis[nd];
  // binary insertion sort (stable)
  for (u32 i = b + 1; i < e; i++) {
    const u32 p = d.order[i];
    const float c = d.cen[3 * (size_t)p + axis];
    u32 lo = b, hi = i;
    while (lo < hi) {
      const u32 mid = (lo + hi) / 2;
      if (c < d.cen[3 * (size_t)d.order[mid] + axis]) hi = mid;
      else lo = mid + 1;
    }
    for (u32 k = i; k > lo; k--) d.order[k] = d.order[k - 1];
    d.order[lo] = p;
  }
}

// Whole subtrees of small nodes (at most kSmall primitives), one wave each,
// with the host builders' recursion (bvh_build.cpp Builder::build /
// FastBuilder::build): the same decisions as the level kernels.  The
// primitives' boxes and centres and the subtree's nodes live in LDS; per node
// the lanes bin the primitives with LDS atomics, each lane evaluates one split
// candidate, and a stable partition by ballots reorders the range.  One global
// atomic reserves the nodes of the subtree.
//
// One thread per subtree (the recursion as the host runs it) was bound by its
// serial chain of dependent scratch and global accesses: 12.6 ms for both trees
// of 100k triangles; a wave per subtree takes 1.1 ms (a rebuild of the scene
// 34.2 -> 21.2 ms).
// 2 kSmall - 1, and some for empty children (boxes whose areas overflow): trees with empty leaves are refused in any
// case, here or when they are emitted
constexpr u32 kSmallNodes = 160;

__device__ __forceinline__ u32 rank_of(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((u32)(m >> 32), __builtin_amdgcn_mbcnt_lo((u32)m, 0u));
}
__device__ __forceinline__ float wave_min(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

struct SmallNodes {
  u32 beg[kSmallNodes], end[kSmallNodes], depth[kSmallNodes], right[kSmallNodes], child[kSmallNodes];
  DBox box[kSmallNodes];
};

// The union of the boxes of positions [b, e), by every lane of the wave.
__device__ DBox wave_union(const float (*s_box)[kSmall], u32 q, u32 b, u32 e) {
  const bool in = threadIdx.x >= b && threadIdx.x < e;
  DBox r = dempty();
  for (int k = 0; k < 3; k++) {
    r.mn[k] = wave_min(in ? s_box[k][q] : r.mn[k]);
    r.mx[k] = wave_max(in ? s_box[3 + k][q] : r.mx[k]);
  }
  return r;
}

__global__ __launch_bounds__(64) void k_small(Dev d) {
  __shared__ float s_box[6][kSmall], s_cen[3][kSmall];
  __shared__ u32 s_prim[kSmall], s_perm[kSmall], s_bins[kMaxSlotWords];
  __shared__ SmallNodes s_n;
  static_assert(kSmall == 64u, "one lane per primitive");
  const u32 root = d.lo + blockIdx.x, lane = threadIdx.x;
  const u32 first = d.nbeg[root], total = d.nend[root] - first;
  if ((d.nflags[root] & kDone) || total > kSmall) return;  // whole wave
  if (lane < total) {
    const u32 p = d.order[first + lane];
    const DBox b = prim_box(d, p);
    s_prim[lane] = p;
    for (int k = 0; k < 3; k++) {
      s_box[k][lane] = b.mn[k];
      s_box[3 + k][lane] = b.mx[k];
      s_cen[k][lane] = d.cen[3 * (size_t)p + k];
    }
  }
  s_perm[lane] = lane;
  if (lane == 0) {
    s_n.beg[0] = 0u;
    s_n.end[0] = total;
    s_n.depth[0] = d.ndepth[root];
    s_n.right[0] = d.nright[root];
    for (int k = 0; k < 3; k++) {
      s_n.box[0].mn[k] = d.nbox[6 * (size_t)root + k];
      s_n.box[0].mx[k] = d.nbox[6 * (size_t)root + 3 + k];
    }
  }
  __syncthreads();
  const u32 K = d.K, axes = d.axes, words = axes * K * 7u;
  u32 count = 1;
  for (u32 id = 0; id < count; id++) {
    const u32 b = s_n.beg[id], e = s_n.end[id], n = e - b, depth = s_n.depth[id];
    if (lane == 0) s_n.child[id] = kInvalid;
    if (depth >= d.max_depth || n <= (d.mode == 0 ? d.bin_size : 1u)) continue;  // utils.rs:20-37
    const bool in = lane >= b && lane < e;
    const u32 q = s_perm[lane];  // below total for a lane in the range
    const DBox box = s_n.box[id];
    // binning parameters of every axis
    float org[3] = {0.0f, 0.0f, 0.0f}, scale[3] = {0.0f, 0.0f, 0.0f};
    int axis0 = 0;
    bool live = true;
    if (d.mode == 0) {
      axis0 = dlongest(box);
      org[0] = box.mn[axis0];
      scale[0] = (box.mx[axis0] - box.mn[axis0]) / (float)K;  // the bins' step
    } else {
      live = false;
      for (int k = 0; k < 3; k++) {
        const float lo = wave_min(in ? s_cen[k][q] : __builtin_inff()), hi = wave_max(in ? s_cen[k][q] : -__builtin_inff());
        const float ext = hi - lo;
        org[k] = lo;
        scale[k] = ext > 0.0f ? (float)K / ext : 0.0f;
        live |= ext > 0.0f;
      }
    }
    auto bin_of = [&](u32 a) {
      return d.mode == 0 ? ref_bin(s_cen[axis0][q], org[0], scale[0], K)
                         : fast_bin(s_cen[a][q], a == 0 ? org[0] : a == 1 ? org[1] : org[2],
                                    a == 0 ? scale[0] : a == 1 ? scale[1] : scale[2], K);
    };
    auto axis_live = [&](u32 a) { return d.mode == 0 || (a == 0 ? scale[0] : a == 1 ? scale[1] : scale[2]) > 0.0f; };
    DBox l = dempty(), r = dempty();
    u32 mid = b, pos = lane;
    bool median = !live;
    double best = __builtin_inf();
    u32 at = 64u;  // the lane of the best candidate
    if (!median) {
      for (u32 w = lane; w < words; w += 64u)
        s_bins[w] = w < axes * K ? 0u : (((w - axes * K) % 6u) < 3u ? kMinInit : kMaxInit);
      __syncthreads();
      if (in)
        for (u32 a = 0; a < axes; a++) {
          if (!axis_live(a)) continue;
          const u32 slot = a * K + bin_of(a);
          atomicAdd(&s_bins[slot], 1u);
          u32 *bk = s_bins + axes * K + 6u * slot;
          for (int k = 0; k < 3; k++) {
            atomicMin(&bk[k], fkey(s_box[k][q]));
            atomicMax(&bk[3 + k], fkey(s_box[3 + k][q]));
          }
        }
      __syncthreads();
      if (d.mode == 0) {
        u32 empty = 0;
        for (u32 k = 0; k < K; k++) empty += s_bins[k] == 0u ? 1u : 0u;
        median = empty == K - 1u;
      }
    }
    if (!median) {
      // lane t evaluates the split of axis t / (K - 1) after bin t % (K - 1)
      const u32 a = lane / (K - 1u), k = lane % (K - 1u);
      double cost = __builtin_inf();
      if (a < axes && axis_live(a)) {
        u32 lc = 0, rc = 0;
        for (u32 w = 0; w < K; w++) {
          const u32 c = s_bins[a * K + w];
          const DBox bb = bin_box(d, s_bins, a * K + w);
          if (w <= k) {
            lc += c;
            dgrow(l, bb);
          } else {
            rc += c;
            dgrow(r, bb);
          }
        }
        if (d.mode == 0) cost = (double)(darea(l) * (float)lc + darea(r) * (float)rc);  // compared as floats: exact
        else if (lc != 0u && lc != n) cost = (double)darea(l) * lc + (double)darea(r) * rc;
        if (!(cost < __builtin_inf())) cost = __builtin_inf();
      }
      // the first strict minimum in (axis, bin) order
      best = cost;
      at = cost < __builtin_inf() ? lane : 64u;
      for (int o = 32; o > 0; o >>= 1) {
        const double c2 = __shfl_xor(best, o, 64);
        const u32 t2 = (u32)__shfl_xor((int)at, o, 64);
        if (c2 < best || (c2 == best && t2 < at)) {
          best = c2;
          at = t2;
        }
      }
      if (d.mode == 1) {
        const double split_cost = d.node_cost + d.prim_cost * best / fmax((double)darea(box), 1e-30);
        if (n <= d.max_leaf && split_cost >= d.prim_cost * n) continue;  // leaf
        if (at == 64u) continue;                                        // unreachable: a live axis splits
        const u32 ba = at / (K - 1u), bk = at % (K - 1u);
        const bool left = in && bin_of(ba) <= bk;
        const unsigned long long ml = __ballot(left), mr = __ballot(in && !left);
        mid = b + (u32)__popcll(ml);
        pos = left ? b + rank_of(ml) : mid + rank_of(mr);
      } else {
        // stable reorder by bin; no finite cost leaves the left child empty
        const u32 w = in ? bin_of(0u) : K;
        u32 off = b;
        for (u32 k2 = 0; k2 < K; k2++) {
          const unsigned long long m = __ballot(w == k2);
          if (w == k2) pos = off + rank_of(m);
          off += (u32)__popcll(m);
          if (at < 64u && k2 <= at) mid = off;
        }
        if (at == 64u) l = r = dempty();
      }
      __syncthreads();
      if (in) s_perm[pos] = q;
    } else {
      mid = b + n / 2u;
      if (d.mode == 0 && lane == 0) {  // stable sort by centre on the longest axis
        for (u32 i = b + 1u; i < e; i++) {
          const u32 p = s_perm[i];
          const float c = s_cen[axis0][p];
          u32 k = i;
          while (k > b && c < s_cen[axis0][s_perm[k - 1u]]) {
            s_perm[k] = s_perm[k - 1u];
            k--;
          }
          s_perm[k] = p;
        }
      }
      __syncthreads();
      const u32 q2 = s_perm[lane];
      l = wave_union(s_box, q2, b, mid);
      r = wave_union(s_box, q2, mid, e);
      at = 0u;
    }
    if (count + 2u > kSmallNodes) {  // only degenerate boxes or options get here: reported
      if (lane == 0) atomicOr(&d.count[2], kErrNodes);
      return;
    }
    if (lane == (at < 64u ? at : 0u)) {
      s_n.child[id] = count;
      s_n.box[count] = l;
      s_n.box[count + 1u] = r;
      for (u32 c = 0; c < 2u; c++) {
        s_n.beg[count + c] = c ? mid : b;
        s_n.end[count + c] = c ? e : mid;
        s_n.depth[count + c] = depth + 1u;
        s_n.right[count + c] = s_n.right[id] + c;
      }
    }
    count += 2u;
    __syncthreads();
  }
  __syncthreads();
  u32 at = 0;
  if (lane == 0 && count > 1u) at = atomicAdd(&d.count[0], count - 1u);
  at = (u32)__shfl((int)at, 0, 64);
  if (count > 1u && at + count - 1u > d.cap) {
    if (lane == 0) atomicOr(&d.count[2], kErrNodes);
    return;
  }
  if (lane < total) d.order[first + lane] = s_prim[s_perm[lane]];
  const u32 geo = d.ngeo[root];
  for (u32 i = lane; i < count; i += 64u) {
    const u32 c = s_n.child[i], g = i == 0u ? root : at + i - 1u;
    d.nchild[g] = c == kInvalid ? kInvalid : at + c - 1u;
    if (c != kInvalid) d.nlc[g] = s_n.end[c] - s_n.beg[c];
    if (i == 0u) {
      d.nflags[g] |= kDone | (c == kInvalid ? 0u : 1u);
      continue;
    }
    const DBox bx = s_n.box[i];
    for (int k = 0; k < 3; k++) {
      d.nbox[6 * (size_t)g + k] = bx.mn[k];
      d.nbox[6 * (size_t)g + 3 + k] = bx.mx[k];
    }
    d.nbeg[g] = first + s_n.beg[i];
    d.nend[g] = first + s_n.end[i];
    d.ndepth[g] = s_n.depth[i];
    d.nright[g] = s_n.right[i];
    d.ngeo[g] = geo;
    d.nflags[g] = kDone | (c == kInvalid ? 0u : 1u);
  }
}

// Partition key of every position: the bin (reference, 4-way stable
// reorder), left / right (fast), or the half (median splits).
__global__ __launch_bounds__(kB) void k_keys(Dev d) {
  const u32 i = blockIdx.x * kB + threadIdx.x;
  if (i > d.n) return;
  uint4 key = make_uint4(0u, 0u, 0u, 0u);
  if (i < d.n) {
    const u32 nd = d.node_of[i];
    if (active(d, nd) && (d.nflags[nd] & 1u)) {
      u32 k;
      if (d.nflags[nd] & 2u) {
        k = i < d.nbeg[nd] + d.nlc[nd] ? 0u : 1u;
      } else {
        const u32 p = d.order[i];
        if (d.mode == 0) {
          const int axis = d.naxis[nd];
          k = ref_bin(d.cen[3 * (size_t)p + axis], d.na[3 * (size_t)nd], d.ns[3 * (size_t)nd], d.K);
        } else {
          const int axis = d.naxis[nd];
          const u32 w = fast_bin(d.cen[3 * (size_t)p + axis], d.na[3 * (size_t)nd + axis], d.ns[3 * (size_t)nd + axis],
                                 d.K);
          k = w <= d.nbest[nd] ? 0u : 1u;
        }
      }
      key.x = k == 0;
      key.y = k == 1;
      key.z = k == 2;
      key.w = k == 3;
    }
  }
  d.keys[i] = key;
}

__device__ __forceinline__ uint4 add4(uint4 a, uint4 b) { return make_uint4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }
__device__ __forceinline__ u32 lane(uint4 a, u32 k) { return k == 0 ? a.x : k == 1 ? a.y : k == 2 ? a.z : a.w; }

// Exclusive scan of keys[0 .. n] in three passes: block sums, one
// workgroup over the block sums, block scans.
constexpr u32 kScanItems = 4;
constexpr u32 kScanTile = kB * kScanItems;

__global__ __launch_bounds__(kB) void k_scan_reduce(Dev d) {
  __shared__ uint4 s[kB];
  const size_t base = (size_t)blockIdx.x * kScanTile;
  uint4 t = make_uint4(0u, 0u, 0u, 0u);
  for (u32 k = 0; k < kScanItems; k++) {
    const size_t i = base + threadIdx.x * kScanItems + k;
    if (i <= d.n) t = add4(t, d.keys[i]);
  }
  s[threadIdx.x] = t;
  __syncthreads();
  for (u32 o = kB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] = add4(s[threadIdx.x], s[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) d.bsum[blockIdx.x] = s[0];
}

__global__ __launch_bounds__(1024) void k_scan_blocks(Dev d, u32 nblocks) {
  __shared__ uint4 s[1024];
  uint4 carry = make_uint4(0u, 0u, 0u, 0u);
  for (u32 base = 0; base < nblocks; base += 1024) {
    const u32 i = base + threadIdx.x;
    const uint4 v = i < nblocks ? d.bsum[i] : make_uint4(0u, 0u, 0u, 0u);
    s[threadIdx.x] = v;
    __syncthreads();
    for (u32 o = 1; o < 1024; o <<= 1) {  // Hillis-Steele inclusive scan
      const uint4 x = threadIdx.x >= o ? s[threadIdx.x - o] : make_uint4(0u, 0u, 0u, 0u);
      __syncthreads();
      s[threadIdx.x] = add4(s[threadIdx.x], x);
      __syncthreads();
    }
    const uint4 incl = s[threadIdx.x];
    if (i < nblocks) d.bsum[i] = make_uint4(carry.x + incl.x - v.x, carry.y + incl.y - v.y, carry.z + incl.z - v.z,
                                             carry.w + incl.w - v.w);
    const uint4 total = s[1023];
    __syncthreads();
    carry = add4(carry, total);
  }
}

__global__ __launch_bounds__(kB) void k_scan_apply(Dev d) {
  __shared__ uint4 s[kB];
  const size_t base = (size_t)blockIdx.x * kScanTile;
  uint4 v[kScanItems], t = make_uint4(0u, 0u, 0u, 0u);
  for (u32 k = 0; k < kScanItems; k++) {
    const size_t i = base + threadIdx.x * kScanItems + k;
    v[k] = i <= d.n ? d.keys[i] : make_uint4(0u, 0u, 0u, 0u);
    t = add4(t, v[k]);
  }
  s[threadIdx.x] = t;
  __syncthreads();
  for (u32 o = 1; o < kB; o <<= 1) {
    const uint4 x = threadIdx.x >= o ? s[threadIdx.x - o] : make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    s[threadIdx.x] = add4(s[threadIdx.x], x);
    __syncthreads();
  }
  uint4 run = add4(d.bsum[blockIdx.x], make_uint4(s[threadIdx.x].x - t.x, s[threadIdx.x].y - t.y,
                                                   s[threadIdx.x].z - t.z, s[threadIdx.x].w - t.w));
  for (u32 k = 0; k < kScanItems; k++) {
    const size_t i = base + threadIdx.x * kScanItems + k;
    if (i <= d.n) d.scan[i] = run;
    run = add4(run, v[k]);
  }
}

// Stable scatter of every position of a split node to its child's range;
// positions of leaves and finished nodes keep their place and leave.
__global__ __launch_bounds__(kB) void k_scatter(Dev d) {
  const u32 i = blockIdx.x * kB + threadIdx.x;
  if (i >= d.n) return;
  const u32 nd = d.node_of[i];
  const u32 p = d.order[i];
  if (!active(d, nd) || !(d.nflags[nd] & 1u)) {
    d.order2[i] = p;
    d.node_of2[i] = kInvalid;
    return;
  }
  const u32 b = d.nbeg[nd], e = d.nend[nd];
  const uint4 key = d.keys[i], sb = d.scan[b], se = d.scan[e], si = d.scan[i];
  u32 k = key.x ? 0u : key.y ? 1u : key.z ? 2u : 3u;
  u32 dest = b + (lane(si, k) - lane(sb, k));
  for (u32 q = 0; q < k; q++) dest += lane(se, q) - lane(sb, q);
  d.order2[dest] = p;
  d.node_of2[dest] = d.nchild[nd] + (dest < b + d.nlc[nd] ? 0u : 1u);
}

// Preorder from one scan.  Every inner node has two children and the
// leaves of a geometry tile its primitive range, so with L(p) the number of
// leaves starting before position p: a subtree holds 2 (L(end) - L(begin)) - 1
// nodes, and a node's preorder index is its depth plus the nodes of every
// subtree left of its path, 2 (L(begin) - L(geometry start)) - r, r being the
// right-child steps on its path.
__global__ void k_leaf_marks(Dev d, u32 total) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  if (!(d.nflags[i] & 1u) && d.nbeg[i] < d.nend[i]) d.keys[d.nbeg[i]] = make_uint4(1u, 0u, 0u, 0u);
}

__global__ void k_clear_keys(Dev d) {
  const u32 i = blockIdx.x * kB + threadIdx.x;
  if (i <= d.n) d.keys[i] = make_uint4(0u, 0u, 0u, 0u);
}

__global__ void k_emit(Dev d, u32 total, const u32 *goff, const u32 *gbase, TreeNode *out) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const u32 g = d.ngeo[i], b = d.nbeg[i], e = d.nend[i];
  const u32 lb = d.scan[b].x, le = d.scan[e].x, l0 = d.scan[goff[g]].x;
  TreeNode t;
  for (int k = 0; k < 3; k++) {
    t.box.mn[k] = d.nbox[6 * (size_t)i + k];
    t.box.mx[k] = d.nbox[6 * (size_t)i + 3 + k];
  }
  t.begin = b - goff[g];
  t.end = e - goff[g];
  t.inner = (d.nflags[i] & 1u) != 0;
  t.size = b < e ? 2u * (le - lb) - 1u : 1u;
  const u32 at = gbase[g] + d.ndepth[i] + 2u * (lb - l0) - d.nright[i];
  if (at >= total) {  // not a full binary tree over tiling leaves: reported, nothing written
    atomicOr(&d.count[2], kErrNodes);
    return;
  }
  out[at] = t;
}

u32 grid_of(size_t n, u32 b = kB) { return (u32)std::max<size_t>(1, (n + b - 1) / b); }

__global__ void k_init_keys(u32 *keys, u32 m) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < (size_t)m * 6; i += (size_t)gridDim.x * blockDim.x)
    keys[i] = (i % 6) < 3 ? kMinInit : kMaxInit;
}

// counts zero, box keys empty, in every slot's first axes * K * 7 words
__global__ void k_init_bins(u32 *bins, u32 m, u32 words, u32 nbins) {
  const size_t total = (size_t)m * words;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
    const u32 slot = (u32)(t / words), w = (u32)(t % words);
    bins[(size_t)slot * kMaxSlotWords + w] = w < nbins ? 0u : (((w - nbins) % 6) < 3 ? kMinInit : kMaxInit);
  }
}

// One root per geometry over its primitive range [off[g], off[g + 1]).
__global__ void k_roots(Dev d, const u32 *off, u32 ngeo) {
  const u32 g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g == 0) {
    d.count[0] = ngeo;
    d.count[1] = 0u;
    d.count[2] = 0u;
    d.count[3] = ngeo;
  }
  if (g >= ngeo) return;
  d.nbeg[g] = off[g];
  d.nend[g] = off[g + 1];
  d.ndepth[g] = 0u;
  d.nchild[g] = kInvalid;
  d.nflags[g] = 0u;
  d.nright[g] = 0u;
  d.ngeo[g] = g;
}

__global__ void k_reset_counts(u32 *count, u32 total) {
  count[0] = total;
  count[1] = 0u;
  count[2] = 0u;
}

struct Buf {
  void *p = nullptr;
  size_t bytes = 0;
  hipError_t reserve(size_t n) {
    if (n <= bytes) return hipSuccess;
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
    hipError_t e = hipMalloc(&p, n);
    if (e == hipSuccess) bytes = n;
    return e;
  }
  ~Buf() {
    if (p) (void)hipFree(p);
  }
};

#define DB_TRY(expr)                     \
  do {                                   \
    hipError_t e_ = (expr);              \
    if (e_ != hipSuccess) return e_;     \
  } while (0)

class Builder final : public DeviceTreeBuilder {
 public:
  explicit Builder(hipStream_t st) : st_(st) {}

  int build(const std::vector<const std::vector<Box> *> &geos, const TreeOptions &ref_opt,
            const FastTreeOptions &fast_opt, std::vector<Tree> &ref, std::vector<Tree> &fast,
            std::string &err) override {
    const u32 rb = ref_opt.bins < 2 ? 4u : ref_opt.bins;
    if (rb > kMaxRefBins) {
      err = "device build supports at most 4 reference SAH bins";
      return RDRT_ERR_CAPACITY;
    }
    if (fast_opt.bins != kFastBins) {
      err = "device build supports 16 fast-tree bins";
      return RDRT_ERR_CAPACITY;
    }
    size_t total = 0;
    for (const auto *g : geos) total += g->size();
    if (total + geos.size() >= (1u << 30)) {
      err = "device build supports fewer than 2^30 primitives per scene";
      return RDRT_ERR_CAPACITY;
    }
    ref.assign(geos.size(), Tree());
    fast.assign(geos.size(), Tree());
    if (geos.empty()) return RDRT_OK;
    if (total == 0) {  // only empty geometries: single empty leaves
      for (size_t g = 0; g < geos.size(); g++) {
        ref[g] = build_tree(*geos[g], ref_opt, 1);
        fast[g] = build_fast_tree(*geos[g], fast_opt, 1);
      }
      return RDRT_OK;
    }
    error_.clear();
    hipError_t e = upload(geos);
    if (e == hipSuccess) e = run(0, ref_opt, fast_opt, ref);
    if (e == hipSuccess) e = run(1, ref_opt, fast_opt, fast);
    if (!error_.empty()) {
      err = "device build does not support this scene: " + error_;
      return RDRT_ERR_CAPACITY;
    }
    if (e != hipSuccess) {
      err = std::string("device build: ") + hipGetErrorString(e);
      return RDRT_ERR_HIP;
    }
    return RDRT_OK;
  }

 private:
  hipStream_t st_;
  Buf pbox_, cen_, order_, order2_, node_of_, node_of2_, keys_, scan_, bsum_, nodes_, bins_, cb_, count_, geo_of_,
      off_, gbase_, emit_;
  Dev d_{};
  size_t cap_nodes_ = 0;
  std::vector<u32> off_h_;  // primitive offset of every geometry (+ total)
  std::string error_;

  hipError_t upload(const std::vector<const std::vector<Box> *> &geos) {
    const u32 ng = (u32)geos.size();
    off_h_.assign(ng + 1, 0u);
    for (u32 g = 0; g < ng; g++) off_h_[g + 1] = off_h_[g] + (u32)geos[g]->size();
    const size_t n = off_h_[ng];
    BigVec<float> h(6 * n);  // every element written below, by geometry in parallel
    BigVec<u32> gof(n);
    host_for(ng, [&](size_t g) {
      for (size_t i = 0; i < geos[g]->size(); i++) {
        const Box &b = (*geos[g])[i];
        const size_t k = off_h_[g] + i;
        std::memcpy(&h[6 * k], b.mn, 12);
        std::memcpy(&h[6 * k + 3], b.mx, 12);
        gof[k] = (u32)g;
      }
    });
    DB_TRY(pbox_.reserve(6 * n * 4));
    DB_TRY(cen_.reserve(3 * n * 4));
    DB_TRY(order_.reserve(n * 4));
    DB_TRY(order2_.reserve(n * 4));
    DB_TRY(node_of_.reserve(n * 4));
    DB_TRY(node_of2_.reserve(n * 4));
    DB_TRY(geo_of_.reserve(n * 4));
    DB_TRY(off_.reserve((ng + 1) * 4));
    DB_TRY(keys_.reserve((n + 1) * 16));
    DB_TRY(scan_.reserve((n + 1) * 16));
    DB_TRY(bsum_.reserve((size_t)(grid_of(n + 1, kScanTile) + 1) * 16));
    DB_TRY(count_.reserve(16));
    cap_nodes_ = 2 * n + ng;  // every geometry a binary tree over its primitives
    // per node: box 6 f; begin, end, depth, child, flags, lc, axis; origin 3 f, step 3 f; best
    DB_TRY(nodes_.reserve(cap_nodes_ * 22 * 4));
    DB_TRY(hipMemcpyAsync(pbox_.p, h.data(), 6 * n * 4, hipMemcpyHostToDevice, st_));
    DB_TRY(hipMemcpyAsync(geo_of_.p, gof.data(), n * 4, hipMemcpyHostToDevice, st_));
    DB_TRY(hipMemcpyAsync(off_.p, off_h_.data(), (ng + 1) * 4, hipMemcpyHostToDevice, st_));
    Dev d{};
    d.n = (u32)n;
    d.pbox = (const float *)pbox_.p;
    d.cen = (float *)cen_.p;
    d.keys = (uint4 *)keys_.p;
    d.scan = (uint4 *)scan_.p;
    d.bsum = (uint4 *)bsum_.p;
    d.count = (u32 *)count_.p;
    d.cap = (u32)cap_nodes_;
    float *f = (float *)nodes_.p;
    d.nbox = f;
    u32 *w = (u32 *)(f + 6 * cap_nodes_);
    d.nbeg = w;
    d.nend = w + cap_nodes_;
    d.ndepth = w + 2 * cap_nodes_;
    d.nchild = w + 3 * cap_nodes_;
    d.nflags = w + 4 * cap_nodes_;
    d.nlc = w + 5 * cap_nodes_;
    d.naxis = (int *)(w + 6 * cap_nodes_);
    d.na = (float *)(w + 7 * cap_nodes_);
    d.ns = (float *)(w + 10 * cap_nodes_);
    d.nbest = w + 13 * cap_nodes_;
    d.nright = w + 14 * cap_nodes_;
    d.ngeo = w + 15 * cap_nodes_;
    d_ = d;
    return hipStreamSynchronize(st_);  // before the host staging arrays go
  }

  hipError_t run(u32 mode, const TreeOptions &ro, const FastTreeOptions &fo, std::vector<Tree> &out) {
    Dev d = d_;
    const size_t n = d.n;
    const u32 ng = (u32)off_h_.size() - 1;
    d.order = (u32 *)order_.p;
    d.order2 = (u32 *)order2_.p;
    d.node_of = (u32 *)node_of_.p;
    d.node_of2 = (u32 *)node_of2_.p;
    d.mode = mode;
    d.K = mode == 0 ? (ro.bins < 2 ? 4u : ro.bins) : kFastBins;
    d.axes = mode == 0 ? 1u : 3u;
    d.max_depth = mode == 0 ? ro.max_depth : fo.max_depth;
    d.bin_size = ro.bin_size;
    d.max_leaf = std::max(1u, std::min(fo.max_leaf, kLeafMaxCount));
    d.node_cost = fo.node_cost;
    d.prim_cost = fo.prim_cost;
    // the roots: one per geometry, boxes the unions of their primitives
    hipLaunchKernelGGL(k_centres, dim3(grid_of(n)), dim3(kB), 0, st_, d, (const u32 *)geo_of_.p);
    hipLaunchKernelGGL(k_roots, dim3(grid_of(ng, 64)), dim3(64), 0, st_, d, (const u32 *)off_.p, ng);
    DB_TRY(cb_.reserve((size_t)ng * 6 * 4));
    u32 *keys = (u32 *)cb_.p;
    d.lo = 0;
    d.m = ng;
    hipLaunchKernelGGL(k_init_keys, dim3(std::min(grid_of((size_t)ng * 6), 4096u)), dim3(kB), 0, st_, keys, ng);
    hipLaunchKernelGGL(k_range_boxes, dim3(grid_of(n)), dim3(kB), 0, st_, d, keys);
    hipLaunchKernelGGL(k_decode_boxes, dim3(grid_of(ng, 64)), dim3(64), 0, st_, d, (const u32 *)keys, 1u);
    u32 lo = 0, m = ng, total = ng;
    while (m > 0) {
      d.lo = lo;
      d.m = m;
      DB_TRY(bins_.reserve((size_t)m * kMaxSlotWords * 4));
      DB_TRY(cb_.reserve((size_t)m * 6 * 4));
      d.bins = (u32 *)bins_.p;
      d.cb = (u32 *)cb_.p;
      const u32 g = grid_of(n), gn = grid_of(m, 64);
      hipLaunchKernelGGL(k_small, dim3(m), dim3(64), 0, st_, d);
      if (mode == 1) {
        hipLaunchKernelGGL(k_init_keys, dim3(std::min(grid_of((size_t)m * 6), 4096u)), dim3(kB), 0, st_, d.cb, m);
        hipLaunchKernelGGL(k_centre_bounds, dim3(g), dim3(kB), 0, st_, d);
      }
      hipLaunchKernelGGL(k_prep, dim3(gn), dim3(64), 0, st_, d);
      const u32 nbins = d.axes * d.K;
      hipLaunchKernelGGL(k_init_bins, dim3(std::min(grid_of((size_t)m * nbins * 7), 8192u)), dim3(kB), 0, st_, d.bins,
                         m, nbins * 7, nbins);
      hipLaunchKernelGGL(k_bins, dim3(g), dim3(kB), 0, st_, d);
      hipLaunchKernelGGL(k_split, dim3(gn), dim3(64), 0, st_, d);
      if (mode == 0) hipLaunchKernelGGL(k_median_sort, dim3(gn), dim3(64), 0, st_, d);
      hipLaunchKernelGGL(k_keys, dim3(grid_of(n + 1)), dim3(kB), 0, st_, d);
      const u32 sb = grid_of(n + 1, kScanTile);
      hipLaunchKernelGGL(k_scan_reduce, dim3(sb), dim3(kB), 0, st_, d);
      hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, st_, d, sb);
      hipLaunchKernelGGL(k_scan_apply, dim3(sb), dim3(kB), 0, st_, d);
      hipLaunchKernelGGL(k_scatter, dim3(g), dim3(kB), 0, st_, d);
      DB_TRY(hipGetLastError());
      u32 counts[4];
      DB_TRY(hipMemcpyAsync(counts, d.count, 16, hipMemcpyDeviceToHost, st_));
      DB_TRY(hipStreamSynchronize(st_));
      if (counts[2]) {
        error_ = counts[2] & kErrMedian ? "a median split of more than 4096 primitives (reference tree)"
                                        : "more nodes than 2n + 1 per geometry (bin_size 0)";
        return hipErrorNotSupported;
      }
      // the nodes that k_small made are finished: no level of theirs
      const u32 next = counts[3], made = counts[0] - next;
      if (counts[1]) {  // children of median splits: boxes are the unions of their ranges
        Dev c = d;
        c.lo = next;
        c.m = made;
        c.node_of = d.node_of2;
        c.order = d.order2;
        DB_TRY(cb_.reserve((size_t)made * 6 * 4));
        u32 *ck = (u32 *)cb_.p;
        hipLaunchKernelGGL(k_init_keys, dim3(std::min(grid_of((size_t)made * 6), 4096u)), dim3(kB), 0, st_, ck, made);
        hipLaunchKernelGGL(k_range_boxes, dim3(g), dim3(kB), 0, st_, c, ck);
        hipLaunchKernelGGL(k_decode_boxes, dim3(grid_of(made, 64)), dim3(64), 0, st_, c, (const u32 *)ck, 2u);
      }
      std::swap(d.order, d.order2);
      std::swap(d.node_of, d.node_of2);
      lo = next;
      m = made;
      total = counts[0];
      hipLaunchKernelGGL(k_reset_counts, dim3(1), dim3(1), 0, st_, d.count, total);
    }
    return download(d, total, out);
  }

  // Preorder nodes of every geometry emitted on the device (k_emit), then
  // one copy of them and of the order to the host, split per geometry
  // (geometry-local primitive indices and ranges).
  hipError_t download(Dev &d, u32 total, std::vector<Tree> &out) {
    const size_t n = d.n;
    const u32 ng = (u32)off_h_.size() - 1;
    hipLaunchKernelGGL(k_clear_keys, dim3(grid_of(n + 1)), dim3(kB), 0, st_, d);
    hipLaunchKernelGGL(k_leaf_marks, dim3(grid_of(total)), dim3(kB), 0, st_, d, total);
    const u32 sb = grid_of(n + 1, kScanTile);
    hipLaunchKernelGGL(k_scan_reduce, dim3(sb), dim3(kB), 0, st_, d);
    hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, st_, d, sb);
    hipLaunchKernelGGL(k_scan_apply, dim3(sb), dim3(kB), 0, st_, d);
    // leaves per geometry -> node counts and bases
    std::vector<uint4> at(ng + 1);
    for (u32 g = 0; g <= ng; g++)
      DB_TRY(hipMemcpyAsync(&at[g], d.scan + off_h_[g], sizeof(uint4), hipMemcpyDeviceToHost, st_));
    DB_TRY(hipStreamSynchronize(st_));
    std::vector<u32> gbase(ng + 1, 0u);
    for (u32 g = 0; g < ng; g++) {
      const u32 leaves = at[g + 1].x - at[g].x;
      gbase[g + 1] = gbase[g] + (leaves ? 2u * leaves - 1u : 1u);
    }
    if (gbase[ng] != total) return hipErrorIllegalState;  // the node count disagrees with the leaves
    DB_TRY(gbase_.reserve((ng + 1) * 4));
    DB_TRY(emit_.reserve((size_t)total * sizeof(TreeNode)));
    DB_TRY(hipMemcpyAsync(gbase_.p, gbase.data(), (ng + 1) * 4, hipMemcpyHostToDevice, st_));
    hipLaunchKernelGGL(k_emit, dim3(grid_of(total)), dim3(kB), 0, st_, d, total, (const u32 *)off_.p,
                       (const u32 *)gbase_.p, (TreeNode *)emit_.p);
    // host copies, filled by the copies below (no zero fill first)
    BigVec<TreeNode> nodes(total);
    BigVec<u32> order(n), depth(total);
    DB_TRY(hipMemcpyAsync(nodes.data(), emit_.p, (size_t)total * sizeof(TreeNode), hipMemcpyDeviceToHost, st_));
    DB_TRY(hipMemcpyAsync(order.data(), d.order, n * 4, hipMemcpyDeviceToHost, st_));
    DB_TRY(hipMemcpyAsync(depth.data(), d.ndepth, (size_t)total * 4, hipMemcpyDeviceToHost, st_));
    BigVec<u32> ngeo(total);
    DB_TRY(hipMemcpyAsync(ngeo.data(), d.ngeo, (size_t)total * 4, hipMemcpyDeviceToHost, st_));
    u32 errs = 0;
    DB_TRY(hipMemcpyAsync(&errs, d.count + 2, 4, hipMemcpyDeviceToHost, st_));
    DB_TRY(hipStreamSynchronize(st_));
    if (errs) return hipErrorIllegalState;
    host_for(ng, [&](size_t g) {
      Tree &t = out[g];
      t.nodes.assign(nodes.begin() + gbase[g], nodes.begin() + gbase[g + 1]);
      t.order.assign(order.begin() + off_h_[g], order.begin() + off_h_[g + 1]);
      for (u32 &p : t.order) p -= off_h_[g];
      t.depth = 0;
    });
    for (u32 i = 0; i < total; i++) out[ngeo[i]].depth = std::max(out[ngeo[i]].depth, depth[i]);
    return hipSuccess;
  }
};

}  // namespace

std::unique_ptr<DeviceTreeBuilder> make_device_tree_builder(hipStream_t stream) {
  return std::unique_ptr<DeviceTreeBuilder>(new Builder(stream));
}

}  // namespace rdrt
