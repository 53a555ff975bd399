// Broad phase: element boxes and a linear BVH (LBVH) for gfx950.
//
// Replaces the reference's incremental AABB tree (AABB.cpp:129-343).  The
// reference's candidate set is "every unordered pair of distinct elements
// whose boxes, inflated by 1e-6, overlap under the closed test"
// (AABB.cpp:10-33, 56-60, 284-343); the tree only fixes the visiting order.
// Here:
//   * k_element_boxes : FP64 static or swept boxes per element (the
//     reference's min/max_{static,moving}_coord, dcollid.cpp:852-932).
//   * k_bounds / k_morton : 30-bit Morton codes of FP32 box centres.
//   * (radix sort of codes, cs_sort.hip)
//   * k_karras        : radix tree over the sorted codes (index tie-break);
//     k_preorder / k_permute : the tree laid out in depth-first pre-order
//     with escape links (ropes) for stackless traversal.
//   * k_refit_tiles / k_refit_top : FP32 boxes of all nodes, rounded outward,
//     so every FP64 overlap is also an FP32 overlap.
//   * k_traverse      : one lane per leaf in Morton order; it starts at its
//     own leaf's rope, so it visits exactly the subtrees after itself in
//     depth-first order (every pair once, no stack); a
//     leaf overlap is confirmed with the exact FP64 boxes, then the
//     reference's early rejects (shared vertex, same rigid surface;
//     dcollid.cpp:762, 805; dcollid3d.cpp:209-214, 257-264, 279-284) run
//     before the pair is appended to the compacted candidate stream.
#include <algorithm>

#include "cs_internal.h"
#include "cs_pairs.h"
#include "cs_tune.h"

namespace cs {

// the box centre of element e into the running bounds m
__device__ inline void centre_bounds(const dbox& b, float m[6]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float c = (float)(0.5 * (b.lo[d] + b.hi[d]));
    m[d] = fminf(m[d], c);
    m[3 + d] = fmaxf(m[3 + d], c);
  }
}

// The bounds of a work-group's threads into its row.  The rows are reduced by
// every work-group of k_morton (no atomics: 6,144 of them on six addresses took
// 50-110 us).
constexpr int BOUNDS_BLOCKS = 128, BOUNDS_THREADS = 512;
template <int THREADS>
__device__ inline void bounds_row(float m[6], float* __restrict__ bounds) {
  __shared__ float s[6][THREADS / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      m[d] = fminf(m[d], __shfl_xor(m[d], o));
      m[3 + d] = fmaxf(m[3 + d], __shfl_xor(m[3 + d], o));
    }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int d = 0; d < 6; ++d) s[d][threadIdx.x >> 6] = m[d];
  __syncthreads();
  if (threadIdx.x < 6) {
    const int d = threadIdx.x;
    float r = s[d][0];
    for (int w = 1; w < THREADS / 64; ++w) r = d < 3 ? fminf(r, s[d][w]) : fmaxf(r, s[d][w]);
    bounds[6 * blockIdx.x + d] = r;
  }
}

// Element boxes (the reference's min/max_{static,moving}_coord,
// dcollid.cpp:852-932), inflated by 1e-6: static boxes into sbox, swept boxes
// into mbox, either may be null.
// m: the bounds of the box centres (of mbox where there is one).
__device__ inline void element_box(const int4* __restrict__ ev, const dvec4* __restrict__ x,
                                   const dvec4* __restrict__ x_old, const dvec4* __restrict__ av,
                                   double dt, int e, dbox* __restrict__ sbox,
                                   dbox* __restrict__ mbox, float m[6]) {
  const int4 t = ev[e];
  const int np = (t.z >= 0) ? 3 : 2;
  const int vid[3] = {t.x, t.y, t.z};
  double lo[2][3], hi[2][3];  // static, swept
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[k][d] = HUGE_VAL;
      hi[k][d] = -HUGE_VAL;
    }
  for (int i = 0; i < np; ++i) {
    const int v = vid[i];
    const dvec4 xo = x_old[v];
    if (mbox) {
      const dvec4 a = av[v];
      const double o[3] = {xo.x, xo.y, xo.z};
      const double n[3] = {xo.x + a.x * dt, xo.y + a.y * dt, xo.z + a.z * dt};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        hi[1][d] = smax(hi[1][d], o[d]);
        hi[1][d] = smax(hi[1][d], n[d]);
        lo[1][d] = smin(lo[1][d], o[d]);
        lo[1][d] = smin(lo[1][d], n[d]);
      }
    }
    if (sbox) {
      // triangles use x_old, bonds use Coords (equal to x_old in the
      // proximity pass; dcollid.cpp:852-860, 892-910)
      dvec4 p = xo;
      if (np != 3) p = x[v];
      const double o[3] = {p.x, p.y, p.z};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        hi[0][d] = smax(o[d], hi[0][d]);
        lo[0][d] = smin(o[d], lo[0][d]);
      }
    }
  }
  dbox* out[2] = {sbox, mbox};
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (!out[k]) continue;
    dbox b;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      b.lo[d] = lo[k][d] - CS_BOX_EPS;
      b.hi[d] = hi[k][d] + CS_BOX_EPS;
    }
    out[k][e] = b;
    if (k == 1 || !mbox) centre_bounds(b, m);
  }
}

__global__ void __launch_bounds__(256) k_element_boxes(const int4* __restrict__ ev,
                                                       const dvec4* __restrict__ x,
                                                       const dvec4* __restrict__ x_old,
                                                       const dvec4* __restrict__ av, double dt, int ne,
                                                       dbox* __restrict__ sbox,
                                                       dbox* __restrict__ mbox,
                                                       float* __restrict__ bounds) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  float m[6] = {3.4e38f, 3.4e38f, 3.4e38f, -3.4e38f, -3.4e38f, -3.4e38f};
  if (e < ne) element_box(ev, x, x_old, av, dt, e, sbox, mbox, m);
  if (bounds) bounds_row<256>(m, bounds);
}

// The bounds of all box centres where the boxes take more work-groups than there
// are rows; up to 32,768 elements k_element_boxes writes the rows itself (one
// launch less, 2.6 us).
__global__ void __launch_bounds__(BOUNDS_THREADS) k_bounds(const dbox* __restrict__ ebox, int ne,
                                                           float* __restrict__ bounds) {
  float m[6] = {3.4e38f, 3.4e38f, 3.4e38f, -3.4e38f, -3.4e38f, -3.4e38f};
  for (int e = blockIdx.x * BOUNDS_THREADS + threadIdx.x; e < ne; e += gridDim.x * BOUNDS_THREADS)
    centre_bounds(ebox[e], m);
  bounds_row<BOUNDS_THREADS>(m, bounds);
}

__device__ inline uint32_t expand_bits10(uint32_t v) {
  v = (v * 0x00010001u) & 0xFF0000FFu;
  v = (v * 0x00000101u) & 0x0F00F00Fu;
  v = (v * 0x00000011u) & 0xC30C30C3u;
  v = (v * 0x00000005u) & 0x49249249u;
  return v;
}

__global__ void __launch_bounds__(256) k_morton(const dbox* __restrict__ ebox, int ne,
                                                const float* __restrict__ bounds, int nbounds,
                                                uint32_t* __restrict__ codes,
                                                uint32_t* __restrict__ ids) {
  __shared__ float s[6][2];
  if (threadIdx.x < BOUNDS_BLOCKS) {  // two wavefronts: the rows of k_bounds
    const int r = min((int)threadIdx.x, nbounds - 1);
    float m[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) m[d] = bounds[6 * r + d];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        m[d] = fminf(m[d], __shfl_xor(m[d], o));
        m[3 + d] = fmaxf(m[3 + d], __shfl_xor(m[3 + d], o));
      }
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int d = 0; d < 6; ++d) s[d][threadIdx.x >> 6] = m[d];
  }
  __syncthreads();
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ne) return;
  const dbox b = ebox[e];
  uint32_t q[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float lo = fminf(s[d][0], s[d][1]), hi = fmaxf(s[3 + d][0], s[3 + d][1]);
    float c = (float)(0.5 * (b.lo[d] + b.hi[d]));
    float ext = hi - lo;
    float u = ext > 0.f ? (c - lo) / ext : 0.5f;
    u = fminf(fmaxf(u, 0.f), 1.f);
    q[d] = (uint32_t)fminf(u * 1024.f, 1023.f);
  }
  codes[e] = (expand_bits10(q[0]) << 2) | (expand_bits10(q[1]) << 1) | expand_bits10(q[2]);
  ids[e] = (uint32_t)e;
}
static_assert(BOUNDS_BLOCKS == 128, "two wavefronts of k_morton");

__device__ inline int lcp_delta(const uint32_t* __restrict__ codes, int n, int i, int j) {
  if (j < 0 || j >= n) return -1;
  const uint32_t a = codes[i], b = codes[j];
  if (a == b) return 32 + __clz((uint32_t)(i ^ j));
  return __clz(a ^ b);
}

// Karras (2012) radix tree, built in construction arrays: internal nodes
// 0..n-2, leaf j is node n-1+j.  The node splitting after leaf g records its
// second child in split_right[g]: that child is what depth-first order
// visits right after any subtree whose last leaf is g (every split position
// 0..n-2 belongs to exactly one internal node).
__global__ void k_karras(const uint32_t* __restrict__ codes, int n, int32_t* __restrict__ kleft,
                         int32_t* __restrict__ kright, int32_t* __restrict__ kparent,
                         int32_t* __restrict__ split_right, int32_t* __restrict__ krmin,
                         int32_t* __restrict__ krmax) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n - 1) return;
  const int d = (lcp_delta(codes, n, i, i + 1) - lcp_delta(codes, n, i, i - 1)) >= 0 ? 1 : -1;
  const int dmin = lcp_delta(codes, n, i, i - d);
  int lmax = 2;
  while (lcp_delta(codes, n, i, i + lmax * d) > dmin) lmax <<= 1;
  int l = 0;
  for (int t = lmax >> 1; t >= 1; t >>= 1)
    if (lcp_delta(codes, n, i, i + (l + t) * d) > dmin) l += t;
  const int j = i + l * d;
  const int dnode = lcp_delta(codes, n, i, j);
  int s = 0;
  int t = l;
  do {
    t = (t + 1) >> 1;
    if (lcp_delta(codes, n, i, i + (s + t) * d) > dnode) s += t;
  } while (t > 1);
  const int gamma = i + s * d + min(d, 0);
  const int lo = min(i, j), hi = max(i, j);
  const int left = (lo == gamma) ? (n - 1) + gamma : gamma;
  const int right = (hi == gamma + 1) ? (n - 1) + gamma + 1 : gamma + 1;
  kleft[i] = left;
  kright[i] = right;
  split_right[gamma] = right;
  krmin[i] = lo;
  krmax[i] = hi;
  kparent[left] = i;
  kparent[right] = i;
  if (i == 0) kparent[0] = -1;
}

// Depth-first (pre-order) position of every construction node: the nodes
// before x are its ancestors and the subtrees left of its path, which hold
// exactly the leaves before x's first leaf a, so pre(x) = 2a + (number of
// left turns from the root to x).  The traversal layout is pre-order: a
// node's first child is the next record and its rope points forward, so a
// walk through the tree touches memory in increasing address order.
__global__ void k_preorder(int n, const int32_t* __restrict__ kleft,
                           const int32_t* __restrict__ kparent, const int32_t* __restrict__ krmin,
                           int32_t* __restrict__ pre) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= 2 * n - 1) return;
  const int a = (x < n - 1) ? krmin[x] : x - (n - 1);
  int left_turns = 0;
  for (int c = x, p = kparent[x]; p >= 0; c = p, p = kparent[p])
    if (kleft[p] == c) ++left_turns;
  pre[x] = 2 * a + left_turns;
}

// scatter the construction tree into the pre-order arrays
__global__ void k_permute(int n, const int32_t* __restrict__ pre, const int32_t* __restrict__ kright,
                          const int32_t* __restrict__ kparent, const int32_t* __restrict__ split_right,
                          const int32_t* __restrict__ krmax,
                          const uint32_t* __restrict__ sorted_ids, bvh_node* __restrict__ nodes,
                          int32_t* __restrict__ parent, int32_t* __restrict__ nright,
                          int32_t* __restrict__ lpre, int32_t* __restrict__ enode) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= 2 * n - 1) return;
  const int p = pre[x];
  const bool internal = x < n - 1;
  const int last = internal ? krmax[x] : x - (n - 1);
  const int rk = (last == n - 1) ? -1 : split_right[last];
  nodes[p].rope = rk < 0 ? -1 : pre[rk];
  parent[p] = kparent[x] < 0 ? -1 : pre[kparent[x]];
  if (internal) {
    nodes[p].left = -1;
    nright[p] = pre[kright[x]];
  } else {
    const int j = x - (n - 1);
    const int e = (int)sorted_ids[j];
    nodes[p].left = e;
    nright[p] = -1;
    lpre[j] = p;
    enode[e] = p;
  }
}

// Refit.  Internal node i of the construction order covers the Morton-sorted
// leaves [krmin, krmax], one end of which is i, so its box is a range minimum /
// maximum over leaf boxes and needs no bottom-up chain (the atomic climb it
// replaces took 150 us from 8,000 leaves on, all of it latency).  A work-group
// holds REFIT_TILE leaf boxes (FP64 boxes rounded outward to FP32) and their
// sparse table (level l: boxes of 2^l leaves) in LDS and answers every node
// inside its tile with two reads; nodes that span tiles are listed and then
// reduced by one wavefront each, over the leaves at both ends and the tile
// boxes between.  Both kernels: 7,938 leaves 153 -> 18 us, 484,530 190 -> 50 us,
// 2.2e6 400 -> under 110 us.
constexpr int REFIT_SHIFT = 8, REFIT_TILE = 1 << REFIT_SHIFT;

struct Box6 {
  float v[6];  // lo, hi
};
__device__ inline Box6 box_empty() { return Box6{{3.4e38f, 3.4e38f, 3.4e38f, -3.4e38f, -3.4e38f, -3.4e38f}}; }
__device__ inline void box_merge(Box6& a, const Box6& b) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    a.v[d] = fminf(a.v[d], b.v[d]);
    a.v[3 + d] = fmaxf(a.v[3 + d], b.v[3 + d]);
  }
}
__device__ inline void box_store(bvh_node* __restrict__ n, const Box6& b) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    n->lo[d] = b.v[d];
    n->hi[d] = b.v[3 + d];
  }
}

__global__ void __launch_bounds__(REFIT_TILE)
    k_refit_tiles(const dbox* __restrict__ ebox, const uint32_t* __restrict__ sorted_ids, int n,
                  bvh_node* __restrict__ nodes, const int32_t* __restrict__ lpre,
                  const int32_t* __restrict__ krmin, const int32_t* __restrict__ krmax,
                  const int32_t* __restrict__ pre, float* __restrict__ tbox,
                  int32_t* __restrict__ top, int* __restrict__ ntop) {
  __shared__ float s[REFIT_SHIFT + 1][6][REFIT_TILE];
  __shared__ int s_cnt, s_base;
  const int t = threadIdx.x, first = blockIdx.x * REFIT_TILE, j = first + t;
  Box6 b = box_empty();
  if (j < n) {
    const dbox d = ebox[sorted_ids[j]];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      b.v[c] = f32_down(d.lo[c]);
      b.v[3 + c] = f32_up(d.hi[c]);
    }
    box_store(nodes + lpre[j], b);
  }
#pragma unroll
  for (int c = 0; c < 6; ++c) s[0][c][t] = b.v[c];
#pragma unroll
  for (int l = 0; l < REFIT_SHIFT; ++l) {  // (past the tile's end: the boxes there are)
    __syncthreads();
    const int u = min(t + (1 << l), REFIT_TILE - 1);
    Box6 o;
#pragma unroll
    for (int c = 0; c < 6; ++c) o.v[c] = s[l][c][u];
    box_merge(b, o);
#pragma unroll
    for (int c = 0; c < 6; ++c) s[l + 1][c][t] = b.v[c];
  }
  __syncthreads();
  if (t < 6) tbox[6 * (size_t)blockIdx.x + t] = s[REFIT_SHIFT][t][0];
  bool span = false;
  if (j < n - 1) {
    const int a = krmin[j], z = krmax[j];
    span = (a >> REFIT_SHIFT) != (z >> REFIT_SHIFT);
    if (!span) {
      const int l = 31 - __clz(z - a + 1), p = a - first, q = z - first + 1 - (1 << l);
      Box6 r;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        r.v[c] = fminf(s[l][c][p], s[l][c][q]);
        r.v[3 + c] = fmaxf(s[l][3 + c][p], s[l][3 + c][q]);
      }
      box_store(nodes + pre[j], r);
    }
  }
  const int slot = block_append(span, ntop, &s_cnt, &s_base);
  if (span) top[slot] = j;
}

__global__ void __launch_bounds__(256)
    k_refit_top(const int32_t* __restrict__ top, const int* __restrict__ ntop,
                const int32_t* __restrict__ krmin, const int32_t* __restrict__ krmax,
                const int32_t* __restrict__ pre, const int32_t* __restrict__ lpre,
                const float* __restrict__ tbox, bvh_node* __restrict__ nodes) {
  const int lane = threadIdx.x & 63, nt = *ntop;
  for (int k = blockIdx.x * 4 + (threadIdx.x >> 6); k < nt; k += gridDim.x * 4) {
    const int i = top[k], a = krmin[i], z = krmax[i];
    const int ta = a >> REFIT_SHIFT, tz = z >> REFIT_SHIFT;
    Box6 b = box_empty();
    auto leaf = [&](int j) {
      const bvh_node m = nodes[lpre[j]];
      box_merge(b, Box6{{m.lo[0], m.lo[1], m.lo[2], m.hi[0], m.hi[1], m.hi[2]}});
    };
    for (int j = a + lane; j < (ta + 1) << REFIT_SHIFT; j += 64) leaf(j);
    for (int j = (tz << REFIT_SHIFT) + lane; j <= z; j += 64) leaf(j);
    for (int q = ta + 1 + lane; q < tz; q += 64) {
      Box6 m;
#pragma unroll
      for (int c = 0; c < 6; ++c) m.v[c] = tbox[6 * (size_t)q + c];
      box_merge(b, m);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      Box6 m;
#pragma unroll
      for (int c = 0; c < 6; ++c) m.v[c] = __shfl_xor(b.v[c], o);
      box_merge(b, m);
    }
    if (lane == 0) box_store(nodes + pre[i], b);
  }
}

// (no short circuit, as f64_overlap below)
__device__ inline bool f32_overlap(const bvh_node& a, const float lo[3], const float hi[3]) {
  return (a.lo[0] <= hi[0]) & (a.hi[0] >= lo[0]) & (a.lo[1] <= hi[1]) & (a.hi[1] >= lo[1]) &
         (a.lo[2] <= hi[2]) & (a.hi[2] >= lo[2]);
}

// AABB::isCollid.  All six comparisons are evaluated (no short circuit), so
// the compiler keeps the box loads together in one round trip instead of
// sinking each component's load behind the previous comparison.
__device__ inline bool f64_overlap(const dbox& a, const dbox& b) {
  return (a.lo[0] <= b.hi[0]) & (a.hi[0] >= b.lo[0]) & (a.lo[1] <= b.hi[1]) &
         (a.hi[1] >= b.lo[1]) & (a.lo[2] <= b.hi[2]) & (a.hi[2] >= b.lo[2]);
}

// Reference early rejects for the canonical orientation (a = hi, b = lo):
// 0 kept, REJ_RIGID same rigid surface, REJ_SHARED a shared vertex.
constexpr int REJ_RIGID = 1, REJ_SHARED = 2;
__device__ inline int pair_reject_kind(int4 ta, int4 tb, uint8_t fa) {
  const bool tri_a = ta.z >= 0, tri_b = tb.z >= 0;
  if (tri_a && tri_b) {
    if (ta.w == tb.w && (fa & EF_RIGID)) return REJ_RIGID;  // same rigid surface
    const int va[3] = {ta.x, ta.y, ta.z}, vb[3] = {tb.x, tb.y, tb.z};
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if (va[i] == vb[k]) return REJ_SHARED;
    return 0;
  }
  if (!tri_a && !tri_b) {
    const int p[4] = {ta.x, ta.y, tb.x, tb.y};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int k = i + 1; k < 4; ++k)
        if (p[i] == p[k]) return REJ_SHARED;
    return 0;
  }
  const int4 T = tri_a ? ta : tb, B = tri_a ? tb : ta;
  const int vt[3] = {T.x, T.y, T.z};
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (vt[i] == B.x || vt[i] == B.y) return REJ_SHARED;
  return 0;
}
__device__ inline bool pair_rejected(int4 ta, int4 tb, uint8_t fa) {
  return pair_reject_kind(ta, tb, fa) != 0;
}
// batched scenes: an element's scene is held in the upper half of its
// surface field (the lower half is the surface's id within the scene)
__device__ inline int scene_of(const int4& t) { return t.w >> 16; }

constexpr int TRAV_BUF = 8;  // pairs buffered per lane before the wavefront writes them

// Full-pass self query.  Lane = one leaf's stackless walk in depth-first order
// after the leaf (every leaf j > i, each subtree once), or a part of it.  What
// bounds it is the chain of dependent node loads of a walk, so walks are cut
// short in two ways, both on one property: a rope walk started at any node x
// visits x's subtree and then the following subtrees, i.e. exactly the nodes
// from x on, so walks over [s0, s1) and [s1, end) find the pairs of the walk
// over [s0, end), each once.
//   * Below TRAV_LANES walks every leaf's walk is cut into 2^lsub sub-ranges
//     from the start (a cut costs up to a tree depth of extra visits).
//   * A walk that reaches TRAV_LONG steps hands the rest of its range to
//     k_traverse_split, where TRAV_SPLIT lanes each walk one sub-range (and hand
//     over once more).  Those of a static obstacle's big faces under a cloth
//     visit tens of thousands of nodes.
// Work-groups are dealt out by the hardware, each XCD one contiguous share of
// the leaves.  Pairs are buffered per lane, written by the wavefront when a
// buffer fills, and at the end with one atomic per work-group: counters in
// memory that every wavefront added to (leaves taken, pairs, candidates) had
// cost more than the walks.  Kernel time with the split rounds, per step,
// against that form: 3,202 elements 120 -> 35 us, 7,938 168 -> 62 us, 138,000 780
// -> 314 us, 484,530 in 64 scenes 1,020 -> 317 us, 2.2e6 3,450 -> 1,460 us.
// TRAV_LONG 128 / 256 / 512: 138,000 elements under strings 314 / 490 / 570 us,
// 130,050 of a crumpled cloth (long walks everywhere) 344 / 287 / 285 us, 2.2e6
// 1,460 / 1,720 / 2,250 us.  TRAV_LANES 131,072 / 262,144: 18,000 elements 167 /
// 139 us.
// DUAL: the boxes are the swept boxes of the first CCD pass; the walk also
// counts the static-box overlaps (the proximity pass's boxes, each inside
// its element's swept box) among the pairs it rejects: a pair with a shared
// vertex always overlaps (both static boxes hold that vertex), a pair on one
// rigid surface is tested.  The kept pairs are tested by k_split_seed, so
// one walk serves both passes.
constexpr int TRAV_STEPS = 16;    // walk steps between checks of the buffers
constexpr int TRAV_LONG = 128;
constexpr int TRAV_SPLIT = 64;

// The rest of one walk: element e over the pre-order nodes [lo, hi), with the
// FP32 box of its leaf.
struct __align__(16) TravItem {
  int e, lo, hi, pad;
  float blo[4], bhi[4];
};
static_assert(sizeof(TravItem) == TRAV_ITEM_BYTES, "TravItem layout");

struct TravArgs {
  const bvh_node* nodes;
  const int32_t* lpre;
  const dbox *ebox, *pbox;
  const int4* ev;
  const uint8_t* eflags;
  int n, scenes;
  int2* pairs;
  int cap;
  int* pair_count;
  unsigned long long *cand_count, *pcand_count;
  TravItem* qout;  // where long walks go (null: they walk on)
  int* qout_n;
  int qcap;
  const int* err;  // not null: no walk when the flag is set
};

struct Walk {
  int e = 0, nd = -1, stop = 0, len = 0;  // element, current node (-1: none), end, steps
  float lo[3] = {0.f, 0.f, 0.f}, hi[3] = {0.f, 0.f, 0.f};
  dbox box{};
  int4 t{};
  uint8_t f = 0;
};

struct WalkOut {
  unsigned long long cand = 0, pcand = 0;
  int nbuf = 0;
};

// The wavefront's walks to their ends.  buf: TRAV_BUF x TRAV_THREADS pairs.
template <bool DUAL>
__device__ __attribute__((always_inline)) inline void run_walks(const TravArgs& A, Walk& w, WalkOut& o,
                                                                int2* __restrict__ buf) {
  const int t = threadIdx.x, lane = t & 63;
  while (__ballot(w.nd >= 0)) {
    for (int step = 0; step < TRAV_STEPS && w.nd >= 0; ++step) {
      if (w.len == TRAV_LONG && A.qout) {  // hand the rest of this walk over
        const int slot = atomicAdd(A.qout_n, 1);
        if (slot < A.qcap) {
          A.qout[slot] = TravItem{w.e, w.nd, w.stop, 0, {w.lo[0], w.lo[1], w.lo[2], 0.f},
                                  {w.hi[0], w.hi[1], w.hi[2], 0.f}};
          w.nd = -1;
          break;
        }
        // (no room: this lane walks on)
      }
      ++w.len;
      const bvh_node node = A.nodes[w.nd];
      const bool over = f32_overlap(node, w.lo, w.hi);
      // an internal node's first child is the next record
      w.nd = over && node.left < 0 ? w.nd + 1 : node.rope;
      if (w.nd >= w.stop) w.nd = -1;
      if (!over || node.left < 0) continue;
      const int e = w.e, e2 = node.left;
      // box, topology and flags in one round trip (the exact overlap test
      // almost always passes where the rounded-out tree box did)
      const dbox ob = A.ebox[e2];
      const int4 ot = A.ev[e2];
      const uint8_t of = A.eflags[e2];
      // (the topology and flags are consumed here so that their loads are
      // issued with the box's, not after the overlap test)
      asm volatile("" ::"v"(ot.x), "v"(ot.y), "v"(ot.z), "v"(ot.w), "v"((int)of));
      if (!f64_overlap(ob, w.box)) continue;
      if (A.scenes && scene_of(ot) != scene_of(w.t)) continue;  // batched scenes never pair up
      ++o.cand;
      const int rk = (e > e2) ? pair_reject_kind(w.t, ot, w.f) : pair_reject_kind(ot, w.t, of);
      if (rk) {
        if constexpr (DUAL)
          if (rk == REJ_SHARED || f64_overlap(A.pbox[e], A.pbox[e2])) ++o.pcand;
        continue;
      }
      buf[o.nbuf * TRAV_THREADS + t] = make_int2(min(e, e2), max(e, e2));
      if (++o.nbuf == TRAV_BUF) break;  // the buffer is written before the walk goes on
    }
    if (__ballot(o.nbuf == TRAV_BUF)) {  // write the wavefront's buffered pairs
      int incl = o.nbuf;
#pragma unroll
      for (int q = 1; q < 64; q <<= 1) {
        const int y = __shfl_up(incl, q);
        if (lane >= q) incl += y;
      }
      int base = 0;
      if (lane == 63) base = atomicAdd(A.pair_count, incl);
      base = __shfl(base, 63) + incl - o.nbuf;
      for (int k = 0; k < o.nbuf; ++k)
        if (base + k < A.cap) A.pairs[base + k] = buf[k * TRAV_THREADS + t];
      o.nbuf = 0;
    }
  }
}

// the rest of the pairs and the counts, one atomic each per work-group (all of
// its threads call it)
template <bool DUAL>
__device__ inline void finish_walks(const TravArgs& A, const WalkOut& o, const int2* __restrict__ buf) {
  constexpr int W = TRAV_THREADS / 64;
  __shared__ unsigned long long s_c[2][W];
  __shared__ int s_n[W], s_base;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  unsigned long long c = o.cand, pc = o.pcand;
  int incl = o.nbuf;
#pragma unroll
  for (int q = 1; q < 64; q <<= 1) {
    const int y = __shfl_up(incl, q);
    if (lane >= q) incl += y;
    c += __shfl_xor(c, q);
    if constexpr (DUAL) pc += __shfl_xor(pc, q);
  }
  if (lane == 63) {
    s_c[0][w] = c;
    s_c[1][w] = pc;
    s_n[w] = incl;
  }
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int q = 0; q < W; ++q) {
    if (q < w) before += s_n[q];
    total += s_n[q];
  }
  if (t < (DUAL ? 2 : 1)) {
    unsigned long long v = 0;
    for (int q = 0; q < W; ++q) v += s_c[t][q];
    if (v) atomicAdd(t == 0 ? A.cand_count : A.pcand_count, v);
  }
  if (t == 64) s_base = total ? atomicAdd(A.pair_count, total) : 0;
  __syncthreads();
  const int base = s_base + before + incl - o.nbuf;
  for (int k = 0; k < o.nbuf; ++k)
    if (base + k < A.cap) A.pairs[base + k] = buf[k * TRAV_THREADS + t];
}

__device__ inline void walk_element(const TravArgs& A, Walk& w) {
  w.box = A.ebox[w.e];
  w.t = A.ev[w.e];
  w.f = A.eflags[w.e];
  w.len = 0;
}

template <bool DUAL>
__global__ void __launch_bounds__(TRAV_THREADS) k_traverse(TravArgs A, int lsub) {
  __shared__ int2 buf[TRAV_BUF * TRAV_THREADS];
  if (A.err && *A.err) return;
  const int nnodes = 2 * A.n - 1;
  const int64_t nw = (int64_t)A.n << lsub;  // walks
  WalkOut o;
  const int share = xcd_block(blockIdx.x, gridDim.x);
  for (int64_t i0 = (int64_t)share * TRAV_THREADS; i0 < nw; i0 += (int64_t)gridDim.x * TRAV_THREADS) {
    const int64_t i = i0 + threadIdx.x;
    Walk w;
    if (i < nw) {
      const bvh_node me = A.nodes[A.lpre[i >> lsub]];
      w.e = me.left;
      walk_element(A, w);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        w.lo[d] = me.lo[d];
        w.hi[d] = me.hi[d];
      }
      w.nd = me.rope;
      w.stop = nnodes;
      if (lsub > 0 && w.nd >= 0) {  // this lane's share of [rope, nnodes)
        const int sub = (int)(i & ((1 << lsub) - 1));
        const int64_t span = nnodes - w.nd;
        w.stop = w.nd + (int)((span * (sub + 1)) >> lsub);
        w.nd += (int)((span * sub) >> lsub);
        if (w.nd >= w.stop) w.nd = -1;
      }
    }
    run_walks<DUAL>(A, w, o, buf);
  }
  finish_walks<DUAL>(A, o, buf);
}

// Split walks: lane g walks sub-range g % TRAV_SPLIT of item g / TRAV_SPLIT.
template <bool DUAL>
__global__ void __launch_bounds__(TRAV_THREADS) k_traverse_split(TravArgs A,
                                                                 const TravItem* __restrict__ qin,
                                                                 const int* __restrict__ qin_n) {
  __shared__ int2 buf[TRAV_BUF * TRAV_THREADS];
  const int64_t total = (int64_t)min(*qin_n, A.qcap) * TRAV_SPLIT;
  if ((int64_t)blockIdx.x * TRAV_THREADS >= total) return;
  WalkOut o;
  for (int64_t g0 = (int64_t)blockIdx.x * TRAV_THREADS; g0 < total;
       g0 += (int64_t)gridDim.x * TRAV_THREADS) {
    const int64_t g = g0 + threadIdx.x;
    Walk w;
    if (g < total) {
      const TravItem it = qin[g / TRAV_SPLIT];
      const int j = (int)(g % TRAV_SPLIT);
      const int64_t span = (int64_t)it.hi - it.lo;
      w.nd = it.lo + (int)(span * j / TRAV_SPLIT);
      w.stop = it.lo + (int)(span * (j + 1) / TRAV_SPLIT);
      if (w.nd >= w.stop) w.nd = -1;
      w.e = it.e;
      walk_element(A, w);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        w.lo[d] = it.blo[d];
        w.hi[d] = it.bhi[d];
      }
    }
    run_walks<DUAL>(A, w, o, buf);
  }
  finish_walks<DUAL>(A, o, buf);
}

// The swept-box pairs of the dual traversal whose static boxes overlap are
// the proximity pass's stream (and are counted with its candidates).  One
// tile of SPLIT_TILE pairs per work-group, one atomic per tile.
constexpr int SPLIT_ITEMS = 16;
constexpr int SPLIT_TILE = 256 * SPLIT_ITEMS;
__global__ void __launch_bounds__(256) k_split_seed(const int2* __restrict__ seed, int n,
                                                    int first, int cap,
                                                    const dbox* __restrict__ pbox,
                                                    int2* __restrict__ prox,
                                                    int* __restrict__ counters) {
  __shared__ int s_off[256];
  __shared__ int s_base;
  const int t = threadIdx.x;
  const int total = counters[CNT_PAIRS];
  if (total > cap) return;  // the stream overflowed: it is walked again
  n = min(n, total);
  const int base_i = first + blockIdx.x * SPLIT_TILE;
  if (base_i >= n) return;
  int2 p[SPLIT_ITEMS];
  uint32_t keep = 0u;
#pragma unroll
  for (int k = 0; k < SPLIT_ITEMS; ++k) {
    const int i = base_i + k * 256 + t;
    p[k] = make_int2(0, 0);
    if (i < n) {
      p[k] = seed[i];
      if (f64_overlap(pbox[p[k].x], pbox[p[k].y])) keep |= 1u << k;
    }
  }
  const int mine = __popc(keep);
  s_off[t] = mine;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {  // inclusive scan of the counts
    const int y = t >= off ? s_off[t - off] : 0;
    __syncthreads();
    s_off[t] += y;
    __syncthreads();
  }
  if (t == 255) {
    s_base = s_off[255] ? atomicAdd(&counters[CNT_PPAIRS], s_off[255]) : 0;
    if (s_off[255])
      atomicAdd(reinterpret_cast<unsigned long long*>(counters + CNT_PCAND64),
                (unsigned long long)s_off[255]);
  }
  __syncthreads();
  int o = s_base + s_off[t] - mine;
#pragma unroll
  for (int k = 0; k < SPLIT_ITEMS; ++k)
    if ((keep >> k) & 1u) prox[o++] = p[k];
}

// ---------------------------------------------------------------------------
// Incremental CCD / impact-zone passes.  Between two passes of one step only
// the average velocities of vertices touched by the last apply or zone update
// change ("dirty" vertices).  A pair whose two elements have no dirty vertex
// keeps its swept boxes, its candidate status and its narrow-phase result
// bit for bit, so the next pass carries those over and only
//   * re-queries dirty elements against the refit tree,
//   * re-runs the narrow phase on pairs that touch a dirty element.
// Candidate counts stay exact: count = previous - (pairs touching dirty
// elements under the previous boxes) + (the same under the new boxes).


// dirty_e[e] = epoch: element has a dirty vertex; list of dirty elements, each
// once.  The dirty vertices are those the last pass changed: the vertices of
// its hits (vlist, nvl of them) and, after a zone pass, the movable members
// of the impact zones (zlist, nzone of them).  Their elements are found
// through the vertex -> element table, one thread per (vertex, MD_SLOTS-th
// element); an exchange on the element's word keeps the first finder.  The
// marks are the number of the marking, so none is cleared (a launch per pass,
// 4 us of about 100, when they were bytes).
constexpr int MD_SLOTS = 8;
__global__ void __launch_bounds__(256) k_mark_dirty(const int32_t* __restrict__ vlist,
                                                    const int* __restrict__ vcount,
                                                    const uint32_t* __restrict__ zlist, int nzone,
                                                    const uint8_t* __restrict__ fixed,
                                                    const int32_t* __restrict__ vadj_ptr,
                                                    const int32_t* __restrict__ vadj,
                                                    uint32_t* __restrict__ dirty_e, uint32_t epoch,
                                                    int32_t* __restrict__ dlist,
                                                    const int32_t* __restrict__ enode,
                                                    uint32_t* __restrict__ dpre,
                                                    uint32_t* __restrict__ rflag,
                                                    int32_t* __restrict__ rlist,
                                                    int* __restrict__ counters) {
  const int nvl = *vcount;
  const long long total = (long long)(nvl + nzone) * MD_SLOTS;
  const long long stride = (long long)gridDim.x * blockDim.x;
  // whole wavefronts iterate together (the appends are per wavefront)
  for (long long t0 = (long long)blockIdx.x * blockDim.x; t0 < total; t0 += stride) {
    const long long t = t0 + threadIdx.x;
    int a = 0, a1 = 0;
    if (t < total) {
      const int k = (int)(t / MD_SLOTS);
      const int v = k < nvl ? vlist[k] : (int)zlist[k - nvl];
      if (k < nvl || !fixed[v]) {
        a = vadj_ptr[v] + (int)(t % MD_SLOTS);
        a1 = vadj_ptr[v + 1];
      }
    }
    for (;; a += MD_SLOTS) {
      const bool live = a < a1;
      if (!__ballot(live)) break;
      int e = 0;
      bool first = false;
      if (live) {
        e = vadj[a];
        first = atomicExch(&dirty_e[e], epoch) != epoch;
      }
      const int slot = wave_append(first, &counters[CNT_DIRTY]);
      bool new_range = false;
      int r = 0;
      if (first) {
        dlist[slot] = e;
        // the leaf, and its QW_RANGE-node range of the pre-order layout
        const int p = enode[e];
        dpre[p] = epoch;
        r = p >> QW_RANGE_SHIFT;
        new_range = atomicExch(&rflag[r], epoch) != epoch;
      }
      const int rs = wave_append(new_range, &counters[CNT_DRANGES]);
      if (new_range) rlist[rs] = r;
    }
  }
}

// Incremental refit by growth.  Between full refits only dirty elements
// change their boxes; each dirty leaf gets its exact new FP32 box and then
// grows its ancestors, stopping at the first one that already contains it.
// Internal boxes only grow (they stay valid bounds, possibly loose, until
// the next full refit); growth uses integer atomics on the float bit
// patterns, so concurrent growers of one node compose.  A plain load that
// sees containment is safe to stop on: a node's box only grows during the
// kernel, and whoever grew it carries the growth further up.
__device__ inline void atomic_min_f32(float* a, float v) {
  if (v >= 0.0f) atomicMin(reinterpret_cast<int*>(a), __float_as_int(v));
  else atomicMax(reinterpret_cast<unsigned int*>(a), __float_as_uint(v));
}
__device__ inline void atomic_max_f32(float* a, float v) {
  if (v >= 0.0f) atomicMax(reinterpret_cast<int*>(a), __float_as_int(v));
  else atomicMin(reinterpret_cast<unsigned int*>(a), __float_as_uint(v));
}

struct GrowArgs {
  const int4* ev;
  const dvec4 *x_old, *av;
  double dt;
  const int32_t* dlist;
  dbox* ebox;
  const int32_t* enode;
  bvh_node* nodes;
  const int32_t* parent;
  int grow;
};

// the dirty elements of work-group `block` of `blocks`
__device__ inline void grow_dirty(const GrowArgs& G, int nd, int block, int blocks) {
  const int4* __restrict__ ev = G.ev;
  const dvec4* __restrict__ x_old = G.x_old;
  const dvec4* __restrict__ av = G.av;
  dbox* __restrict__ ebox = G.ebox;
  bvh_node* nodes = G.nodes;
  const double dt = G.dt;
  for (int k = block * blockDim.x + threadIdx.x; k < nd; k += blocks * blockDim.x) {
    const int e = G.dlist[k];
    // the element's new swept box
    const int4 t = ev[e];
    const int np = (t.z >= 0) ? 3 : 2;
    const int vid[3] = {t.x, t.y, t.z};
    double blo[3] = {HUGE_VAL, HUGE_VAL, HUGE_VAL};
    double bhi[3] = {-HUGE_VAL, -HUGE_VAL, -HUGE_VAL};
    for (int i = 0; i < np; ++i) {
      const dvec4 xo = x_old[vid[i]];
      const dvec4 a = av[vid[i]];
      const double o[3] = {xo.x, xo.y, xo.z};
      const double nn[3] = {xo.x + a.x * dt, xo.y + a.y * dt, xo.z + a.z * dt};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        bhi[d] = smax(bhi[d], o[d]);
        bhi[d] = smax(bhi[d], nn[d]);
        blo[d] = smin(blo[d], o[d]);
        blo[d] = smin(blo[d], nn[d]);
      }
    }
    dbox b;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      b.lo[d] = blo[d] - CS_BOX_EPS;
      b.hi[d] = bhi[d] + CS_BOX_EPS;
    }
    ebox[e] = b;
    if (!G.grow) continue;
    // the leaf exactly, its ancestors grown
    const int leaf = G.enode[e];
    float lo[3], hi[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = f32_down(b.lo[d]);
      hi[d] = f32_up(b.hi[d]);
      nodes[leaf].lo[d] = lo[d];
      nodes[leaf].hi[d] = hi[d];
    }
    for (int node = G.parent[leaf]; node >= 0; node = G.parent[node]) {
      const bvh_node c = nodes[node];
      if ((c.lo[0] <= lo[0]) & (c.lo[1] <= lo[1]) & (c.lo[2] <= lo[2]) & (c.hi[0] >= hi[0]) &
          (c.hi[1] >= hi[1]) & (c.hi[2] >= hi[2]))
        break;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if (lo[d] < c.lo[d]) atomic_min_f32(&nodes[node].lo[d], lo[d]);
        if (hi[d] > c.hi[d]) atomic_max_f32(&nodes[node].hi[d], hi[d]);
      }
    }
  }
}

// Query of every dirty element against the whole tree.  A pair of two dirty
// elements is taken from the one earlier in Morton order.  emit = 0: count
// only (previous boxes, into CNT_OLD64); emit = 1: count into CNT_NEW64 and
// append non-rejected pairs to qpairs.
//
// One wavefront per QW_RANGE-node range of the pre-order layout that holds dirty
// leaves: the range's dirty leaves are neighbours in Morton order, so the
// union of their boxes is small.  The wavefront descends the tree breadth
// first with that union box, collects the leaves the union box overlaps, and
// each lane then tests its own element against them with the exact boxes.  A
// frontier or leaf list too large for LDS falls back to one stackless walk per
// lane.  A zone pass has a few hundred ranges of about 27 leaves each in a tree
// 27 levels deep, so the steps of the descent, a dependent load each, bound the
// kernel.  A step follows chains of up to QW_CHAIN first children, so there are
// about half as many steps as levels.  Query and growth per step (87 passes at
// 1024 x 1024, 33 at 256 x 256, 8 with many ranges on a wavy 256 x 256 sheet):
// 3.95, 1.10, 0.92 ms one level at a time, 3.60, 0.98, 0.80 with chains of 2,
// 3.40, 0.94, 0.81 with 4, 3.66, 1.00, 0.99 with 8.
constexpr int QW_CHAIN = 4;    // records of one first-child chain read at a time
constexpr int QW_FCAP = 1024;  // frontier nodes of one level
constexpr int QW_LCAP = 1024;  // leaves collected by one range

// advances the length of the query's own stream, or (count CNT_PAIRS) that of the
// pair stream and with it the query's count
__device__ inline int add_pairs(int* __restrict__ counters, int count, int n) {
  if (count == CNT_QPAIRS) return atomicAdd(&counters[CNT_QPAIRS], n);
  static_assert(CNT_PAIRS % 2 == 0 && CNT_QPAIRS == CNT_PAIRS + 1, "one 64-bit word");
  return (int)(uint32_t)atomicAdd((unsigned long long*)&counters[CNT_PAIRS],
                                  (unsigned long long)n | (unsigned long long)n << 32);
}

__device__ inline void flush_pairs(int2* buf, int nbuf, int2* __restrict__ qpairs, int qcap,
                                   int* __restrict__ counters, int count) {
  // exclusive scan of nbuf over the wavefront, one atomic per wavefront
  const int lane = threadIdx.x & 63;
  int incl = nbuf;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o);
    if (lane >= o) incl += y;
  }
  const int total = __shfl(incl, 63);
  if (total == 0) return;
  int base = 0;
  if (lane == 63) base = add_pairs(counters, count, total);
  base = __shfl(base, 63) + incl - nbuf;
  for (int q = 0; q < nbuf; ++q)
    if (base + q < qcap) qpairs[base + q] = buf[q * 64 + lane];
}

__global__ void __launch_bounds__(64) k_query_ranges(
    const bvh_node* __restrict__ nodes, const int32_t* __restrict__ nright,
    const dbox* __restrict__ ebox, const int4* __restrict__ ev,
    const uint8_t* __restrict__ eflags, const uint32_t* __restrict__ dirty_e,
    const uint32_t* __restrict__ dpre, uint32_t epoch, const int32_t* __restrict__ rlist, int npre, int emit,
    int scenes, int snap, int exact,
    int2* __restrict__ qpairs, int qcap, int count, int* __restrict__ counters) {
  __shared__ int32_t fr[2][QW_FCAP];
  __shared__ int2 lv[QW_LCAP];  // (pre-order index, element)
  // the range's dirty elements (the queries), compacted: box and pre-order
  // index in one 64 B record (one LDS round trip per query), the rest apart
  struct QueryRec {
    dbox b;
    int32_t si, pad[3];
  };
  __shared__ QueryRec qr[64];
  __shared__ int4 qt[64];
  __shared__ int32_t qe[64];
  __shared__ uint8_t qf[64];
  __shared__ int2 buf[TRAV_BUF * 64];
  const int lane = threadIdx.x;
  const int nr = counters[CNT_DRANGES];
  unsigned long long cand = 0;
  // the counts carried into the pass, before the narrow phase appends
  if (snap && blockIdx.x == 0 && lane < 4) counters[CNT_SNAP + lane] = counters[lane];
  // ranges in block order: the first nr blocks are busy, and the hardware's
  // round-robin placement spreads them over all XCDs
  for (int ri = blockIdx.x; ri < nr; ri += gridDim.x) {
    const int si = QW_RANGE * rlist[ri] + lane;  // this lane's node
    bvh_node me{};
    bool act = false;
    if (lane < QW_RANGE && si < npre) {
      me = nodes[si];
      act = dpre[si] == epoch;
    }
    dbox mb{};
    int4 mt{};
    uint8_t mf = 0;
    int e = -1;
    float ulo[3] = {3.4e38f, 3.4e38f, 3.4e38f}, uhi[3] = {-3.4e38f, -3.4e38f, -3.4e38f};
    if (act) {
      e = me.left;
      mb = ebox[e];
      mt = ev[e];
      mf = eflags[e];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        ulo[d] = me.lo[d];
        uhi[d] = me.hi[d];
      }
    }
#pragma unroll
    for (int o = QW_RANGE / 2; o > 0; o >>= 1)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        ulo[d] = fminf(ulo[d], __shfl_xor(ulo[d], o));
        uhi[d] = fmaxf(uhi[d], __shfl_xor(uhi[d], o));
      }
#pragma unroll
    for (int d = 0; d < 3; ++d) {  // (the lanes past the range hold empty boxes)
      ulo[d] = __shfl(ulo[d], 0);
      uhi[d] = __shfl(uhi[d], 0);
    }
    // Breadth-first descent with the union box.  A node's first child is the
    // next record, so QW_CHAIN lanes take a frontier node and the records
    // behind it: as far as the boxes overlap they go down the chain of first
    // children, and only second children (and what follows the last record)
    // wait for the next step.
    if (lane == 0) fr[0][0] = 0;
    __syncthreads();
    int cur = 0, nfr = 1, nlv = 0;
    bool overflow = false;
    const uint64_t below = (1ull << lane) - 1ull;
    while (nfr > 0) {
      int nnext = 0;
      for (int b = 0; b < nfr; b += 64 / QW_CHAIN) {
        const int i = b + lane / QW_CHAIN, j = lane % QW_CHAIN;
        bool ov = false, inner = false;
        int node = 0, c2 = 0, left = -1;
        if (i < nfr) node = fr[cur][i] + j;
        if (i < nfr && node < npre) {
          const bvh_node N = nodes[node];
          c2 = nright[node];
          left = N.left;
          inner = left < 0;
          ov = f32_overlap(N, ulo, uhi);
        }
        // reached: every record before this one of the four is gone down from
        const uint32_t before = (1u << j) - 1u;
        const uint32_t down = (uint32_t)(__ballot(ov && inner) >> (lane - j));
        const bool reached = ov && (down & before) == before;
        const uint64_t ml = __ballot(reached && !inner), mi = __ballot(reached && inner);
        const uint64_t mc = __ballot(reached && inner && j == QW_CHAIN - 1);
        if (reached && !inner) {
          const int q = nlv + __popcll(ml & below);
          if (q < QW_LCAP) lv[q] = make_int2(node, left);
        }
        if (reached && inner) {
          const int q = nnext + __popcll(mi & below) + __popcll(mc & below);
          if (q < QW_FCAP) fr[cur ^ 1][q] = c2;
          if (j == QW_CHAIN - 1 && q + 1 < QW_FCAP) fr[cur ^ 1][q + 1] = node + 1;
        }
        nlv += __popcll(ml);
        nnext += __popcll(mi) + __popcll(mc);
      }
      __syncthreads();
      if (nlv > QW_LCAP || nnext > QW_FCAP) {
        overflow = true;
        break;
      }
      cur ^= 1;
      nfr = nnext;
    }
    int nbuf = 0;
    // a box-overlapping pair of query element qel and element e2
    auto take = [&](int qel, const int4& qtop, uint8_t qfl, int e2, const int4& ot, uint8_t of) {
      if (scenes && scene_of(ot) != scene_of(qtop)) return;  // batched scenes never pair up
      ++cand;
      if (!emit) return;
      const bool rej = (qel > e2) ? pair_rejected(qtop, ot, qfl) : pair_rejected(ot, qtop, of);
      if (rej) return;
      const int2 pr = make_int2(min(qel, e2), max(qel, e2));
      if (nbuf < TRAV_BUF) {
        buf[nbuf * 64 + lane] = pr;
        ++nbuf;
      } else {
        const int slot = add_pairs(counters, count, 1);
        if (slot < qcap) qpairs[slot] = pr;
      }
    };
    if (!overflow) {
      // lanes hold the collected leaves, 64 at a time; the queries are
      // broadcast from LDS
      const uint64_t am = __ballot(act);
      const int na = __popcll(am);
      if (act) {
        const int q = __popcll(am & below);
        qr[q].b = mb;
        qr[q].si = si;
        qt[q] = mt;
        qe[q] = e;
        qf[q] = mf;
      }
      __syncthreads();
      for (int b = 0; b < nlv; b += 64) {
        const bool have = b + lane < nlv;
        int j = -1, e2 = 0;
        dbox ob{};
        int4 ot{};
        uint8_t of = 0, od = 0;
        if (have) {
          const int2 L = lv[b + lane];
          j = L.x;
          e2 = L.y;
          ob = ebox[e2];
          ot = ev[e2];
          of = eflags[e2];
          od = dirty_e[e2] == epoch;
        }
        // overlaps first (a bit per query), rejects and output afterwards
        uint64_t hits = 0;
#pragma unroll 2
        for (int q = 0; q < na; ++q) {
          const QueryRec Q = qr[q];
          // a pair of two dirty elements is taken from the one earlier in
          // pre-order; the overlap test without branches (AABB::isCollid)
          const bool hit = (j != Q.si) & !(od && j < Q.si) &
                           (ob.lo[0] <= Q.b.hi[0]) & (ob.hi[0] >= Q.b.lo[0]) &
                           (ob.lo[1] <= Q.b.hi[1]) & (ob.hi[1] >= Q.b.lo[1]) &
                           (ob.lo[2] <= Q.b.hi[2]) & (ob.hi[2] >= Q.b.lo[2]);
          hits |= (uint64_t)(have && hit) << q;
        }
        while (hits) {
          const int q = __builtin_ctzll(hits);
          hits &= hits - 1;
          take(qe[q], qt[q], qf[q], e2, ot, of);
        }
      }
    } else if (act) {
      // stackless walk from the root with this lane's leaf box
      int nd = 0;
      while (nd >= 0) {
        const bvh_node node = nodes[nd];
        if (!f32_overlap(node, me.lo, me.hi)) {
          nd = node.rope;
          continue;
        }
        if (node.left < 0) {  // internal: its first child is the next record
          ++nd;
          continue;
        }
        const int j = nd;
        nd = node.rope;
        const int e2 = node.left;
        if (j == si) continue;
        const bool od = dirty_e[e2] == epoch;
        if (od && j < si) continue;  // counted from e2
        if (!f64_overlap(ebox[e2], mb)) continue;
        take(e, mt, mf, e2, ev[e2], eflags[e2]);
      }
    }
    if (emit) flush_pairs(buf, nbuf, qpairs, qcap, counters, count);
    __syncthreads();
  }
  unsigned long long c = cand;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (exact && lane == 0 && c)
    atomicAdd((unsigned long long*)(counters + (emit ? CNT_NEW64 : CNT_OLD64)), c);
}

__global__ void k_clear_counters(uint64_t mask, int* __restrict__ counters) {
  clear_counters(mask, counters);
}

// carry clean pairs of the previous pass
constexpr int CARRY_ITEMS = 16;
__global__ void __launch_bounds__(256) k_carry_pairs(const int2* __restrict__ prev, int n,
                                                     const uint32_t* __restrict__ dirty_e,
                                                     uint32_t epoch, int2* __restrict__ cur, int cap,
                                                     int* __restrict__ counters) {
  __shared__ int s_off[256];
  __shared__ int s_base;
  const int t = threadIdx.x;
  const int base_i = blockIdx.x * 256 * CARRY_ITEMS;
  int2 p[CARRY_ITEMS];
  bool keep[CARRY_ITEMS];
  int nk = 0;
#pragma unroll
  for (int q = 0; q < CARRY_ITEMS; ++q) {
    const int i = base_i + q * 256 + t;
    keep[q] = false;
    if (i < n) {
      p[q] = prev[i];
      keep[q] = dirty_e[p[q].x] != epoch && dirty_e[p[q].y] != epoch;
    }
    nk += keep[q] ? 1 : 0;
  }
  s_off[t] = nk;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int add = (t >= off) ? s_off[t - off] : 0;
    __syncthreads();
    s_off[t] += add;
    __syncthreads();
  }
  if (t == 255) s_base = s_off[255] ? atomicAdd(&counters[CNT_PAIRS], s_off[255]) : 0;
  __syncthreads();
  int o = s_base + s_off[t] - nk;
#pragma unroll
  for (int q = 0; q < CARRY_ITEMS; ++q)
    if (keep[q]) {
      if (o < cap) cur[o] = p[q];
      ++o;
    }
}

struct CarryArgs {
  const hit_rec* hits_prev;
  const int4* hp_prev;
  int nhits, nhp;
  const uint32_t* dirty_e;
  uint32_t epoch;
  hit_rec* hits;
  uint64_t* hkey;
  int hit_cap, hb;
  int4* hp;
  int hp_cap, zone;
  const int4* ev;
  const int32_t* vbody;
  ZoneList Z;
};

// Between the marking of the dirty elements and their query: the first work-groups
// carry the clean hits (with their sort keys) and hit pairs of the previous
// pass over and merge the impact zones of the latter (union order does not
// change the partition), the others give the dirty elements their new boxes.
// One launch: the four that it replaces took 10.6 (growth), 4.4, 3.4 and
// 1.6 us, each alone on the card.
__global__ void __launch_bounds__(256) k_grow_carry(GrowArgs G, CarryArgs C, int bhits, int bhp,
                                                    int* __restrict__ counters) {
  __shared__ int s_cnt, s_base;
  if ((int)blockIdx.x < bhits) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool keep = false;
    uint64_t key = 0;
    if (i < C.nhits) {
      key = C.hits_prev[i].key;
      const int lo = (int)(key >> 36), hi = (int)((key >> 8) & 0xFFFFFFFull);
      keep = C.dirty_e[lo] != C.epoch && C.dirty_e[hi] != C.epoch;
    }
    const int slot = block_append(keep, &counters[CNT_HITS], &s_cnt, &s_base);
    if (keep && slot < C.hit_cap) {
      C.hits[slot] = C.hits_prev[i];
      C.hkey[slot] = hit_sort_key(key, C.hb);
    }
  } else if ((int)blockIdx.x < bhits + bhp) {
    const int i = (blockIdx.x - bhits) * blockDim.x + threadIdx.x;
    int4 r = make_int4(0, 0, 0, 0);
    bool keep = false;
    if (i < C.nhp) {
      r = C.hp_prev[i];
      keep = C.dirty_e[r.x] != C.epoch && C.dirty_e[r.y] != C.epoch;
    }
    const int slot = block_append(keep, &counters[CNT_HIT_PAIRS], &s_cnt, &s_base);
    if (keep && slot < C.hp_cap) C.hp[slot] = r;
    if (keep && C.zone) hp_union(r, C.ev, C.vbody, C.Z);
  } else {
    const int b = bhits + bhp;
    grow_dirty(G, counters[CNT_DIRTY], blockIdx.x - b, gridDim.x - b);
  }
}

hipError_t launch_mark_dirty(hipStream_t st, DevState& S, const int* vcount, int nzone) {
  if (++S.dirty_epoch == 0) {  // after 2^32 - 1 markings the old numbers come again
    const size_t npre = 2 * (size_t)S.ne - 1;
    CS_HIP_RET(hipMemsetAsync(S.dirty_e, 0, sizeof(uint32_t) * (size_t)S.ne, st));
    CS_HIP_RET(hipMemsetAsync(S.dpre, 0, sizeof(uint32_t) * npre, st));
    CS_HIP_RET(hipMemsetAsync(S.rflag, 0, sizeof(uint32_t) * ((npre + QW_RANGE - 1) / QW_RANGE), st));
    S.dirty_epoch = 1;
  }
  // grid for a typical list; longer lists are walked grid-stride
  hipLaunchKernelGGL(k_mark_dirty, dim3(std::min((MD_SLOTS * S.nv + 255) / 256, 256)), dim3(256),
                     0, st, S.vlist, vcount, S.zlist, nzone, S.fixed, S.vadj_ptr, S.vadj,
                     S.dirty_e, S.dirty_epoch, S.dlist, S.leaf_of, S.dpre, S.rflag, S.rlist,
                     S.counters);
  return hipGetLastError();
}

void launch_clear_counters(hipStream_t st, DevState& S, uint64_t mask) {
  hipLaunchKernelGGL(k_clear_counters, dim3(1), dim3(64), 0, st, mask, S.counters);
}

void launch_grow_carry(hipStream_t st, DevState& S, double dt, int nhits_prev, int nhp_prev,
                       int zone) {
  if (S.ne == 0) return;
  const GrowArgs G{S.ev, S.x_old, S.av, dt, S.dlist, S.ebox, S.leaf_of, S.nodes, S.parent,
                   S.ne >= 2 ? 1 : 0};
  const CarryArgs C{S.hits_prev, S.hp_prev, nhits_prev, nhp_prev, S.dirty_e, S.dirty_epoch, S.hits, S.hkey,
                    S.hit_cap, hit_id_bits(S), S.hp, S.hp_cap, zone, S.ev, S.vbody, zone_list(S)};
  const int bh = (nhits_prev + 255) / 256, bp = (nhp_prev + 255) / 256;
  // growth: grid for a typical dirty list; longer lists are walked grid-stride
  hipLaunchKernelGGL(k_grow_carry, dim3(bh + bp + std::min((S.ne + 255) / 256, 512)), dim3(256), 0,
                     st, G, C, bh, bp, S.counters);
}

void launch_query_dirty(hipStream_t st, DevState& S, int emit, int snap, int count, int exact) {
  if (S.ne < 2) return;
  const int npre = 2 * S.ne - 1;
  hipLaunchKernelGGL(k_query_ranges, dim3(query_grid(S.ne, S.tune_query)), dim3(64), 0, st,
                     S.nodes, S.nright, S.ebox, S.ev, S.eflags, S.dirty_e, S.dpre, S.dirty_epoch, S.rlist, npre,
                     emit, S.nscene > 1, snap, exact, count == CNT_PAIRS ? S.pairs : S.qpairs,
                     count == CNT_PAIRS ? S.pair_cap : S.qpair_cap, count, S.counters);
}

void launch_carry_pairs_from(hipStream_t st, DevState& S, const int2* src, int n) {
  if (n > 0)
    hipLaunchKernelGGL(k_carry_pairs, dim3((n + 256 * CARRY_ITEMS - 1) / (256 * CARRY_ITEMS)), dim3(256), 0, st,
                       src, n, S.dirty_e, S.dirty_epoch, S.pairs, S.pair_cap, S.counters);
}

// ---------------------------------------------------------------------------
void launch_element_boxes(hipStream_t st, const DevState& S, double dt, dbox* sbox, dbox* mbox) {
  const int ne = S.ne;
  if (ne == 0) return;
  const int nb = (ne + 255) / 256;
  hipLaunchKernelGGL(k_element_boxes, dim3(nb), dim3(256), 0, st, S.ev, S.x, S.x_old, S.av, dt, ne,
                     sbox, mbox, nb <= BOUNDS_BLOCKS ? S.bounds : nullptr);
}

hipError_t build_bvh(hipStream_t st, DevState& S) {
  const int n = S.ne;
  if (n == 0) return hipSuccess;
  int nb = (n + 255) / 256;  // rows that k_element_boxes wrote
  if (nb > BOUNDS_BLOCKS) {
    nb = std::min(BOUNDS_BLOCKS, (n + BOUNDS_THREADS - 1) / BOUNDS_THREADS);
    hipLaunchKernelGGL(k_bounds, dim3(nb), dim3(BOUNDS_THREADS), 0, st, S.ebox, n, S.bounds);
  }
  hipLaunchKernelGGL(k_morton, dim3((n + 255) / 256), dim3(256), 0, st, S.ebox, n, S.bounds, nb,
                     S.mcode, S.mid);
  bool in_tmp = false;
  CS_HIP_RET(radix_sort_u32(st, S.mcode, S.mid, S.mcode_tmp, S.mid_tmp, S.sort_hist, S.scan_part, n,
                            30, &in_tmp));
  S.sorted_codes = in_tmp ? S.mcode_tmp : S.mcode;
  S.sorted_ids = in_tmp ? S.mid_tmp : S.mid;
  if (n == 1) {  // a single leaf: node 0
    bvh_node leaf{};
    leaf.left = 0;
    leaf.rope = -1;
    const int32_t zero = 0, none = -1;
    CS_HIP_RET(hipMemcpyAsync(S.nodes, &leaf, sizeof(leaf), hipMemcpyHostToDevice, st));
    CS_HIP_RET(hipMemcpyAsync(S.parent, &none, sizeof(int32_t), hipMemcpyHostToDevice, st));
    CS_HIP_RET(hipMemcpyAsync(S.lpre, &zero, sizeof(int32_t), hipMemcpyHostToDevice, st));
    CS_HIP_RET(hipMemcpyAsync(S.leaf_of, &zero, sizeof(int32_t), hipMemcpyHostToDevice, st));
    CS_HIP_RET(hipStreamSynchronize(st));  // host sources above live on this stack frame
  } else {
    const int nn = 2 * n - 1;
    // (every split position 0 .. n - 2 belongs to one node: split_right is written whole)
    hipLaunchKernelGGL(k_karras, dim3((n - 1 + 255) / 256), dim3(256), 0, st, S.sorted_codes, n,
                       S.kleft, S.kright, S.kparent, S.split_right, S.krmin, S.krmax);
    hipLaunchKernelGGL(k_preorder, dim3((nn + 255) / 256), dim3(256), 0, st, n, S.kleft, S.kparent,
                       S.krmin, S.pre);
    hipLaunchKernelGGL(k_permute, dim3((nn + 255) / 256), dim3(256), 0, st, n, S.pre, S.kright,
                       S.kparent, S.split_right, S.krmax, S.sorted_ids, S.nodes, S.parent,
                       S.nright, S.lpre, S.leaf_of);
  }
  return hipGetLastError();
}

// (the caller has zeroed CNT_TMP, the number of nodes that span tiles)
hipError_t refit_bvh(hipStream_t st, DevState& S) {
  const int n = S.ne;
  if (n == 0) return hipSuccess;
  const int tiles = (n + REFIT_TILE - 1) / REFIT_TILE;
  hipLaunchKernelGGL(k_refit_tiles, dim3(tiles), dim3(REFIT_TILE), 0, st, S.ebox, S.sorted_ids, n,
                     S.nodes, S.lpre, S.krmin, S.krmax, S.pre, S.tbox, S.top, S.counters + CNT_TMP);
  if (tiles > 1)
    hipLaunchKernelGGL(k_refit_top, dim3(std::min(tiles, 2048)), dim3(256), 0, st, S.top,
                       S.counters + CNT_TMP, S.krmin, S.krmax, S.pre, S.lpre, S.tbox, S.nodes);
  return hipGetLastError();
}

size_t refit_tile_count(int n) { return (size_t)(n + REFIT_TILE - 1) / REFIT_TILE; }

// (the caller has zeroed the item counts of the split rounds, CNT_TSPLIT)
void launch_traverse(hipStream_t st, DevState& S, int2* out, int cap, const dbox* pbox,
                     bool check) {
  const int n = S.ne;
  if (n < 2) return;
  const int lsub = traverse_cuts(n), blocks = traverse_grid(n, S.num_cus, S.tune_trav);
  TravItem* q0 = reinterpret_cast<TravItem*>(S.tq);
  TravItem* q1 = q0 + TRAV_QCAP;
  int* n0 = S.counters + CNT_TSPLIT;
  TravArgs A{S.nodes, S.lpre, S.ebox, pbox, S.ev, S.eflags, n, S.nscene > 1, out, cap,
             S.counters + CNT_PAIRS, (unsigned long long*)(S.counters + CNT_CAND64),
             (unsigned long long*)(S.counters + CNT_PCAND64), q0, n0, TRAV_QCAP,
             check ? S.counters + CNT_ERR : nullptr};
  TravArgs A1 = A, A2 = A;
  A1.qout = q1;
  A1.qout_n = n0 + 1;
  A2.qout = nullptr;
  A2.qout_n = nullptr;
  // where a share of the tree has no more nodes than a walk may take, no walk is
  // handed over and the rounds for them are not launched (up to 4,095 elements)
  const bool rounds = ((2 * (int64_t)n) >> lsub) + 1 > TRAV_LONG;
  if (!rounds) A.qout = nullptr;
  auto go = [&](auto main, auto split) {
    hipLaunchKernelGGL(main, dim3(blocks), dim3(TRAV_THREADS), 0, st, A, lsub);
    if (!rounds) return;
    hipLaunchKernelGGL(split, dim3(4 * S.num_cus), dim3(TRAV_THREADS), 0, st, A1,
                       (const TravItem*)q0, (const int*)n0);
    hipLaunchKernelGGL(split, dim3(4 * S.num_cus), dim3(TRAV_THREADS), 0, st, A2,
                       (const TravItem*)q1, (const int*)(n0 + 1));
  };
  if (pbox) go(k_traverse<true>, k_traverse_split<true>);
  else go(k_traverse<false>, k_traverse_split<false>);
}

void launch_split_seed(hipStream_t st, DevState& S, int first, int n) {
  if (n <= first) return;
  hipLaunchKernelGGL(k_split_seed, dim3((n - first + SPLIT_TILE - 1) / SPLIT_TILE), dim3(256), 0, st,
                     S.pairs_seed, n, first, S.pair_cap, S.pbox, S.pairs, S.counters);
}

}  // namespace cs
