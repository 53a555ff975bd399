// Element pairs, their sub-tests and the impact-zone union-find, as the narrow
// phase and the carried hit pairs of incremental passes use them.
#pragma once
#include "cs_internal.h"

namespace cs {

// local point indices of sub-test s.  kind: 0 tri-tri (A 0..2, B 3..5),
// 1 tri-bond (tri 0..2, bond 3..4), 2 bond-bond (A 0..1, B 2..3)
__device__ inline void subtest_points(int kind, int s, int ccd, int q[4], bool* is_pt) {
  if (kind == 0) {
    if (s < 6) {
      const int k = s / 3, i = s - 3 * k;
      // proximity: k=0 triangle B, point A[i]; CCD: k=0 triangle A, point B[i]
      const bool tri_is_a = (k == 0) == (ccd != 0);
      const int tb = tri_is_a ? 0 : 3, pb = tri_is_a ? 3 : 0;
      q[0] = tb; q[1] = tb + 1; q[2] = tb + 2; q[3] = pb + i;
      *is_pt = true;
    } else {
      const int i = (s - 6) / 3, j = (s - 6) - 3 * i;
      q[0] = i; q[1] = (i + 1) % 3; q[2] = 3 + j; q[3] = 3 + (j + 1) % 3;
      *is_pt = false;
    }
  } else if (kind == 1) {
    if (s < 2) {
      q[0] = 0; q[1] = 1; q[2] = 2; q[3] = 3 + s;
      *is_pt = true;
    } else {
      const int i = s - 2;
      q[0] = i; q[1] = (i + 1) % 3; q[2] = 3; q[3] = 4;
      *is_pt = false;
    }
  } else {
    q[0] = 0; q[1] = 1; q[2] = 2; q[3] = 3;
    *is_pt = false;
  }
}

__device__ inline int uf_load(int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline int uf_find(int* uf, int x) {
  for (;;) {
    const int p = uf_load(&uf[x]);
    if (p == x) return x;
    const int gp = uf_load(&uf[p]);
    if (gp == p) return p;
    atomicCAS(&uf[x], p, gp);  // path halving; parents only decrease
    x = gp;
  }
}
__device__ inline void uf_union(int* uf, int a, int b) {
  for (;;) {
    a = uf_find(uf, a);
    b = uf_find(uf, b);
    if (a == b) return;
    if (a < b) { const int t = a; a = b; b = t; }
    if (atomicCAS(&uf[a], a, b) == a) return;  // larger root under smaller
  }
}

// zone membership: list each vertex once per step, the first time it is an
// endpoint of a union of two distinct vertices
struct ZoneList {
  int* uf;
  int* mark;
  uint32_t* list;
  int* count;
};
__device__ inline void zone_touch(const ZoneList& Z, int v) {
  if (__hip_atomic_load(&Z.mark[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return;
  if (atomicExch(&Z.mark[v], 1) == 0) Z.list[atomicAdd(Z.count, 1)] = (uint32_t)v;
}
__device__ inline void zone_union(const ZoneList& Z, int a, int b) {
  if (a == b) return;
  zone_touch(Z, a);
  zone_touch(Z, b);
  uf_union(Z.uf, a, b);
}
// createImpZone(pts, 4, NO) (dcollid.cpp:473-484): every pair of the four
// points not holding a movable point is merged, which joins all non-movable
// points of the sub-test; they are merged through the first of them
__device__ inline void zone_merge4(const ZoneList& Z, const int32_t* vbody, const int p[4]) {
  bool ok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) ok[i] = !(vbody && vbody[p[i]] >= 0);
  int hub = -1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (!ok[i]) continue;
    if (hub < 0) hub = p[i];
    else zone_union(Z, hub, p[i]);
  }
}

// vertices of an element pair (canonical orientation: A = hi, B = lo) and
// its kind: 0 tri-tri (15 sub-tests), 1 tri-bond (5), 2 bond-bond (1)
__device__ inline void pair_points(int2 pr, const int4* __restrict__ ev, int* A, int* B, int* kind,
                                   int* nsub, int g[6]) {
  *A = pr.y;
  *B = pr.x;
  const int4 ta = ev[*A], tb = ev[*B];
  const bool tri_a = ta.z >= 0, tri_b = tb.z >= 0;
  if (tri_a && tri_b) {
    *kind = 0; *nsub = 15;
    g[0] = ta.x; g[1] = ta.y; g[2] = ta.z; g[3] = tb.x; g[4] = tb.y; g[5] = tb.z;
  } else if (tri_a || tri_b) {
    const int4 T = tri_a ? ta : tb, Bd = tri_a ? tb : ta;
    *kind = 1; *nsub = 5;
    g[0] = T.x; g[1] = T.y; g[2] = T.z; g[3] = Bd.x; g[4] = Bd.y; g[5] = Bd.y;
  } else {
    *kind = 2; *nsub = 1;
    g[0] = ta.x; g[1] = ta.y; g[2] = tb.x; g[3] = tb.y; g[4] = tb.y; g[5] = tb.y;
  }
}

// impact-zone merges of a hit pair carried from the previous pass (lo, hi, hit
// mask, first hit): the points of every sub-test from the first hit onward
__device__ inline void hp_union(const int4& r, const int4* __restrict__ ev, const int32_t* vbody,
                                const ZoneList& Z) {
  int A, B, kind, nsub, g[6];
  pair_points(make_int2(r.x, r.y), ev, &A, &B, &kind, &nsub, g);
  for (int s = r.w; s < nsub; ++s) {
    int q[4];
    bool is_pt;
    subtest_points(kind, s, 1, q, &is_pt);
    const int p4[4] = {g[q[0]], g[q[1]], g[q[2]], g[q[3]]};
    zone_merge4(Z, vbody, p4);
  }
}

inline ZoneList zone_list(DevState& S) {
  return ZoneList{S.uf, S.zmark, S.zlist, S.counters + CNT_ZLIST};
}

}  // namespace cs
