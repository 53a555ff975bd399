// Host-side plan of the banded strain-limit sweep (plain C++, no HIP).
//
// reduceSuperelast (dcollid.cpp:486-596) sweeps the non-rigid elements in
// element order, in place, up to ten times.  The plan cuts that order into
// `nband` contiguous bands; a task (band, sweep) is run by one work-group
// that keeps the velocities of the vertices in use in LDS:
//   * levels: an element's level is above those of all earlier elements that
//     share a vertex with it, so the elements of one level share no vertex and
//     a vertex meets its elements in level order;
//   * a step of a band: up to STRAIN_STEP_SLOTS of its elements of one level
//     (one lane each), steps in level order;
//   * an import: a vertex enters the band's LDS before its first step there,
//     an export: it leaves after its last step there.  A vertex's visits of
//     one sweep lie in bands of ascending index (bands are contiguous in
//     element order), so its value travels from band to band and, from the
//     last one, to the first band of the next sweep.
// Task (b, k) publishes the level below which all its steps are done and
// exported.  An import waits for one such level: that of the vertex's last
// visit in its previous band (same sweep, a lower band) or, in the vertex's
// first band, that of its last visit in the previous sweep.  Both kinds of
// dependency point to a task earlier in the order (sweep, band), so the tasks
// can run concurrently, and any number of them at a time, without deadlock
// if they are started in that order.
#pragma once
#include <algorithm>
#include <cstdint>
#include <cstring>
#include <limits>
#include <vector>

namespace cs {

constexpr int STRAIN_STEP_SLOTS = 64;   // elements of a step (lanes of a wavefront)
constexpr int STRAIN_GROUP = 4;         // steps whose imports are fetched together
constexpr int STRAIN_IMPORT_WAVES = 2;   // wavefronts fetching imports, group by group in turn
constexpr int STRAIN_AHEAD = 4;          // groups the imports may run ahead of the sweep
constexpr int STRAIN_MAX_BANDS = 64;
constexpr int STRAIN_VERT_BYTES = 56;
constexpr int STRAIN_LDS_VERTS = 2560;  // vertices of a task's LDS window (140 KB of the 160)

// one element of a step, 32 B: rest lengths of edges (0,1), (1,2), (2,0), the
// LDS places of its vertices, its vertex count
struct StrainRec {
  double L0[3];
  uint16_t place[3];
  uint16_t np;
};
struct StrainImport {
  uint32_t v, place;
};
// imports of a group of steps, and the levels they wait for (-1: none): of
// lower bands in the same sweep, of this and higher bands in the previous one;
// the group's records
struct StrainGroup {
  int32_t imp0, imp1, need_same, need_prev, rec0, rec1;
};
struct StrainExport {
  uint32_t v;
  uint32_t place;  // bit 31: the vertex's last visit of the sweep
  int32_t step;    // step of the band after which it leaves
  int32_t pad;
};

// The records of all steps one after another, so that a step takes the room of
// its elements (rows of STRAIN_STEP_SLOTS took 2 KB each, 2 GB for one string of
// 10^6 bonds).  Read as rows: element i % STRAIN_STEP_SLOTS of step
// i / STRAIN_STEP_SLOTS, vertex count 0 where the step has fewer elements.
struct StrainRows {
  std::vector<StrainRec> packed;     // (+ STRAIN_STEP_SLOTS unused ones at the end)
  std::vector<int32_t> first{0};     // [steps + 1] first record of each step
  size_t size() const { return (first.size() - 1) * STRAIN_STEP_SLOTS; }
  int32_t at(size_t i) const { return first[i / STRAIN_STEP_SLOTS] + (int32_t)(i % STRAIN_STEP_SLOTS); }
  const StrainRec& operator[](size_t i) const {
    static const StrainRec none{};
    return at(i) < first[i / STRAIN_STEP_SLOTS + 1] ? packed[(size_t)at(i)] : none;
  }
};

struct StrainPlan {
  int nband = 0, n_levels = 0, cap = 0;   // cap: LDS places of the largest window
  int64_t nvert = 0;                      // vertices of the elements planned
  std::vector<int32_t> step_ptr;          // [nband + 1] steps of each band
  std::vector<int32_t> step_level;        // [steps + 64]
  StrainRows rec;                         // [steps][STRAIN_STEP_SLOTS]
  std::vector<int32_t> grp_ptr;           // [nband + 1] groups of each band
  std::vector<StrainGroup> grp;           // [groups]
  std::vector<StrainImport> imp;
  std::vector<int32_t> exp_ptr;           // [nband + 1]
  std::vector<StrainExport> exp;          // (+ 64 unused entries at the end)
  std::vector<int32_t> lo_ptr, lo;        // lower bands a band's imports come from
  std::vector<int32_t> up_ptr, up;        // bands (of the previous sweep) likewise
  std::vector<int64_t> slot;              // [ne] element -> index into rec, -1 rigid
  size_t steps() const { return step_ptr.empty() ? 0 : (size_t)step_ptr.back(); }
};

// Levels of the non-rigid elements (-1: rigid): earliest levels, then each
// vertex's first visit raised to at most W levels below its last one,
// repeated until nothing moves (W starts at the largest valence - 1 and
// doubles when a pass limit is hit; without convergence the earliest levels
// are kept).  The earliest levels of a row-major grid let the first columns
// run ~1000 levels ahead of their last visit, which would keep every vertex
// in use for the whole sweep; raised, a vertex's visits span 5 levels and the
// number of levels stays.  ev: four ints per element (v0, v1, v2 or -1, -).
// Returns the number of levels.
inline int strain_levels(int nv, int ne, const int* ev, const uint8_t* rigid, std::vector<int>& lev) {
  lev.assign((size_t)std::max(ne, 1), -1);
  auto np_of = [&](int e) { return ev[4 * (size_t)e + 2] >= 0 ? 3 : 2; };
  auto vtx = [&](int e, int k) { return ev[4 * (size_t)e + k]; };
  std::vector<int> valence((size_t)nv, 0);
  int nsched = 0;
  for (int e = 0; e < ne; ++e) {
    if (rigid[e]) continue;
    ++nsched;
    for (int k = 0; k < np_of(e); ++k) valence[vtx(e, k)]++;
  }
  if (nsched == 0) return 0;
  const int maxval = *std::max_element(valence.begin(), valence.end());
  std::vector<int> lv((size_t)nv), last((size_t)nv);
  std::vector<uint8_t> seen((size_t)nv);
  bool converged = false;
  for (int W = std::max(1, maxval - 1); W <= 64 && !converged; W *= 2) {
    for (int e = 0; e < ne; ++e) lev[e] = rigid[e] ? -1 : 0;
    std::fill(last.begin(), last.end(), -1);
    for (int pass = 0; pass < 16; ++pass) {
      bool changed = false;
      std::fill(lv.begin(), lv.end(), -1);
      std::fill(seen.begin(), seen.end(), 0);
      for (int e = 0; e < ne; ++e) {
        if (rigid[e]) continue;
        int l = lev[e];
        for (int k = 0; k < np_of(e); ++k) {
          const int v = vtx(e, k);
          l = std::max(l, lv[v] + 1);
          if (!seen[v]) l = std::max(l, last[v] - W);
        }
        if (l != lev[e]) {
          lev[e] = l;
          changed = true;
        }
        for (int k = 0; k < np_of(e); ++k) {
          lv[vtx(e, k)] = l;
          seen[vtx(e, k)] = 1;
        }
      }
      last = lv;
      if (!changed) {
        converged = true;
        break;
      }
    }
  }
  if (!converged) {  // earliest levels
    std::fill(lv.begin(), lv.end(), -1);
    for (int e = 0; e < ne; ++e) {
      if (rigid[e]) continue;
      int l = 0;
      for (int k = 0; k < np_of(e); ++k) l = std::max(l, lv[vtx(e, k)] + 1);
      lev[e] = l;
      for (int k = 0; k < np_of(e); ++k) lv[vtx(e, k)] = l;
    }
  }
  int L = 0;
  for (int e = 0; e < ne; ++e) L = std::max(L, lev[e] + 1);
  return L;
}

// Bands for `nsched` elements on `n_levels` levels: about 20 elements of a
// band on a level.  A step costs the same for 1 and for 64 elements, and a
// band's tasks start a few steps after the band below, so few, full bands are
// good; but the imports of a step are fetched by the same work-group, and past
// ~30 of them they no longer hide behind the step.  Sweep times at 8 / 16 / 32 /
// 48 elements: 64 x 64 cloth 0.41 / 0.39 / 0.35 / 0.35 ms, 256 x 256 cloth 1.25
// / 1.18 / 1.18 / 1.89 ms, 1024 x 1024 cloth with 2,000 strings 3.0 / 2.5 / 2.6
// / 4.1 ms.
inline int strain_band_count(int64_t nsched, int n_levels) {
  const int64_t b = (nsched + 20ll * n_levels - 1) / (20ll * std::max(n_levels, 1));
  int n = (int)std::min<int64_t>(std::max<int64_t>(b, 1), STRAIN_MAX_BANDS);
  if (n > 8) n = (n + 7) & ~7;  // a band's tasks then tend to share an XCD
  return n;
}

// Whether the banded sweeps are the better ones of a plan that fits, or all sweeps
// in one work-group (k_strain_pipe).  Where many vertices are met by many bands, a
// band begins when the ones below it are nearly over: the bands of all sweeps run
// one after another, and their steps last as long as their imports.  An order
// with locality imports a vertex 1.0 to 2.2 times a sweep (rows, columns, radial,
// Morton; tiles of 16), elements in random order 2.6 times (24 x 24) and more.
// Kernel ms, banded / one work-group, with many / few edges over the limit:
//   imports  mesh                                 many          few
//   1.0      64 x 64 by rows                      0.41 / 1.54   0.27 / 0.85
//   2.1      256 x 256, shuffled tiles of 16      1.45 / 4.63   1.27 / 1.79
//   2.1      32 x 32, shuffled within 1,024       0.31 / 0.35   0.28 / 0.17
//   2.2      512 x 512, shuffled tiles of 16      11.8 / 15.3   11.7 / 2.4
//   2.9      128 x 128, shuffled tiles of 4       4.8 / 1.2     4.8 / 0.28
//   3.7      128 x 128, shuffled within 4,096     1.42 / 1.02   1.38 / 0.28
//   5.7      160 x 160 in random order            11.2 / 1.4    11.2 / 0.31
// A sweep of few steps cannot cost much in bands, and a mesh with every edge over the
// limit gains: 24 x 24 in random order (44 steps) 0.34 / 0.22 and 0.32 / 0.14, but
// the whole step of one with every edge over it 0.59 / 1.00 ms.
inline bool strain_plan_pays(const StrainPlan& P) {
  return 10 * (int64_t)P.imp.size() <= 24 * P.nvert || P.steps() <= 64;
}

// Chains: long schedules with few elements on a level (single strings, strips).
// The bands' steps are made whether or not an element is evaluated, 0.25 us each,
// while the one-work-group sweep goes to the levels with something to do, at some 4 us
// an iteration.  With most bonds over the limit the bands are four times faster, with
// two of 30,000 eight times slower; so a chain is laid out for both, and the number of
// elements over the limit before the sweeps decides at every step (one host wait more,
// 10 us).  Whole step in us, one work-group / bands, by moved points (one puts one
// or two bonds over the limit):
//   open string of 1,000     5: 188 / 401       50: 777 / 443
//   open, 30,000             2: 403 / 6,520     150: 1,580 / 6,690   1,500: 13,100 / 8,000
//   closed, 1,000            2: 1,040 / 2,210   50: 4,590 / 2,340
//   closed, 30,000           2: 27,100 / 59,900 150: 101,000 / 59,600
// The sweeps of a closed string follow each other one by one (one in flight), so an
// element costs more there.  Up to 512 levels the difference is below the wait; above
// 65,536 the one-work-group sweep cannot skip.
constexpr int STRAIN_CHAIN_LEVELS = 512, STRAIN_SKIP_LEVELS = 65536;
inline bool strain_is_chain(int64_t nsched, int n_levels) {
  return n_levels > STRAIN_CHAIN_LEVELS && n_levels <= STRAIN_SKIP_LEVELS && nsched <= 8ll * n_levels;
}
inline bool strain_few(int64_t over, int64_t nsched, bool one_in_flight) {
  return over > 0 && over * (one_in_flight ? 256 : 64) < nsched;
}

// Microseconds after which a wait of a task means that the plan is broken.  A
// task may wait for everything before it: where a vertex's visits span all levels
// (a ring of bonds, a fan) sweep k only begins when sweep k - 1 is nearly over, and
// bands can depend on each other in the same way.  A step takes 0.2 to 1 us, its
// imports and exports included about 2, so 5 for each step of each sweep.
inline int64_t strain_wait_us(int64_t steps, int sweeps) { return 2000000 + 5 * steps * sweeps; }

// Whole components much shorter than the schedule (strings, small pieces) are
// moved to other levels, first fit: at most STRAIN_SHIFT_WIDTH elements of the
// band their first element lies in on any level they occupy (the fewest where
// none fits).  Left at their earliest levels, 1000 strings of a band would all
// be in use at once and overflow its window.
constexpr int STRAIN_SHIFT_WIDTH = 32;
inline void strain_shift_components(int nv, const int* ev, const std::vector<int32_t>& sched,
                                    int nband, int n_levels, std::vector<int>& lev) {
  auto np_of = [&](int e) { return ev[4 * (size_t)e + 2] >= 0 ? 3 : 2; };
  std::vector<int32_t> uf((size_t)nv);
  for (int v = 0; v < nv; ++v) uf[v] = v;
  auto find = [&](int32_t v) {
    while (uf[v] != v) v = uf[v] = uf[uf[v]];
    return v;
  };
  for (int32_t e : sched)
    for (int k = 1; k < np_of(e); ++k) {
      const int32_t a = find(ev[4 * (size_t)e]), c = find(ev[4 * (size_t)e + k]);
      if (a != c) uf[std::max(a, c)] = std::min(a, c);
    }
  std::vector<int32_t> lo((size_t)nv, std::numeric_limits<int32_t>::max()), hi((size_t)nv, -1);
  for (int32_t e : sched) {
    const int32_t r = find(ev[4 * (size_t)e]);
    lo[r] = std::min(lo[r], lev[e]);
    hi[r] = std::max(hi[r], lev[e]);
  }
  auto is_short = [&](int32_t r) { return 2 * (hi[r] - lo[r] + 1) <= n_levels; };
  // load[band][level] of the elements that stay; elements of each short component
  const int64_t ns = (int64_t)sched.size();
  std::vector<std::vector<int32_t>> load((size_t)nband);
  std::vector<std::vector<int32_t>> member;
  std::vector<int32_t> comp((size_t)nv, -1), cband;
  for (int64_t i = 0; i < ns; ++i) {
    const int32_t e = sched[i], r = find(ev[4 * (size_t)e]);
    const int b = (int)(((i + 1) * nband - 1) / ns);
    if (!is_short(r)) {
      if (load[b].empty()) load[b].assign((size_t)n_levels, 0);
      load[b][lev[e]]++;
      continue;
    }
    if (comp[r] < 0) {
      comp[r] = (int32_t)member.size();
      member.emplace_back();
      cband.push_back(b);
    }
    member[comp[r]].push_back(e);
  }
  std::vector<int32_t> hist;
  for (size_t c = 0; c < member.size(); ++c) {
    const int32_t r = find(ev[4 * (size_t)member[c][0]]);
    const int len = hi[r] - lo[r] + 1, range = n_levels - len;
    hist.assign((size_t)len, 0);
    for (int32_t e : member[c]) hist[lev[e] - lo[r]]++;
    auto& ld = load[cband[c]];
    if (ld.empty()) ld.assign((size_t)n_levels, 0);
    const int step = std::max(1, range / 256);
    int best = 0, best_max = std::numeric_limits<int32_t>::max();
    for (int o = 0; o <= range && best_max > STRAIN_SHIFT_WIDTH; o += step) {
      int m = 0;
      for (int j = 0; j < len && m < best_max; ++j) m = std::max(m, ld[o + j] + hist[j]);
      if (m < best_max) {
        best_max = m;
        best = o;
      }
    }
    for (int j = 0; j < len; ++j) ld[best + j] += hist[j];
    for (int32_t e : member[c]) lev[e] += best - lo[r];
  }
}

// The plan with `nband` bands; false when a band's vertex window does not fit
// STRAIN_LDS_VERTS (the caller tries more bands or another method).
inline bool strain_build_plan(int nv, int ne, const int* ev, const uint8_t* rigid,
                              const double* len0 /* [ne][4] */, std::vector<int> lev,
                              int n_levels, int nband, StrainPlan& P) {
  P = StrainPlan();
  P.nband = nband;
  P.n_levels = n_levels;
  auto np_of = [&](int e) { return ev[4 * (size_t)e + 2] >= 0 ? 3 : 2; };
  auto vtx = [&](int e, int k) { return ev[4 * (size_t)e + k]; };
  std::vector<int32_t> sched;
  for (int e = 0; e < ne; ++e)
    if (!rigid[e]) sched.push_back(e);
  const int64_t ns = (int64_t)sched.size();
  P.slot.assign((size_t)std::max(ne, 1), -1);
  strain_shift_components(nv, ev, sched, nband, n_levels, lev);
  // level and band of every vertex's last visit of a sweep
  std::vector<int32_t> vlast((size_t)nv, -1), vband((size_t)nv, -1);
  auto band_begin = [&](int b) { return (size_t)(ns * b / nband); };
  for (int b = 0; b < nband; ++b)
    for (size_t i = band_begin(b); i < band_begin(b + 1); ++i)
      for (int k = 0; k < np_of(sched[i]); ++k) {
        vlast[vtx(sched[i], k)] = lev[sched[i]];
        vband[vtx(sched[i], k)] = b;
      }
  for (int v = 0; v < nv; ++v) P.nvert += vband[v] >= 0;
  std::vector<int32_t> pband((size_t)nv, -1), plevel((size_t)nv, -1);  // previous band's last visit
  std::vector<int32_t> stamp((size_t)nv, -1), fstep((size_t)nv), lstep((size_t)nv), place((size_t)nv);
  std::vector<int32_t> order, cnt((size_t)n_levels + 1), touched;
  std::vector<std::vector<int32_t>> bystep;
  P.step_ptr.push_back(0);
  P.grp_ptr.push_back(0);
  P.exp_ptr.push_back(0);
  P.lo_ptr.push_back(0);
  P.up_ptr.push_back(0);
  for (int b = 0; b < nband; ++b) {
    const size_t i0 = band_begin(b), i1 = band_begin(b + 1);
    // the band's elements by level (element order within a level)
    std::fill(cnt.begin(), cnt.end(), 0);
    for (size_t i = i0; i < i1; ++i) cnt[(size_t)lev[sched[i]] + 1]++;
    std::vector<int32_t> lvl_of_step;
    for (int l = 0; l < n_levels; ++l) {
      for (int c = 0; c < cnt[(size_t)l + 1]; c += STRAIN_STEP_SLOTS) lvl_of_step.push_back(l);
      cnt[(size_t)l + 1] += cnt[l];
    }
    order.resize(i1 - i0);
    {
      std::vector<int32_t> at(cnt.begin(), cnt.end() - 1);
      for (size_t i = i0; i < i1; ++i) order[at[lev[sched[i]]]++] = sched[i];
    }
    const int nstep = (int)lvl_of_step.size();
    const size_t step0 = P.steps();
    // slots, and each vertex's first and last step in the band
    touched.clear();
    {
      int st = -1, fill = STRAIN_STEP_SLOTS, cur = -1;
      for (int32_t e : order) {
        if (lev[e] != cur || fill == STRAIN_STEP_SLOTS) {
          ++st;
          fill = 0;
          cur = lev[e];
          P.rec.first.push_back(P.rec.first.back());
        }
        P.slot[e] = (int64_t)((step0 + st) * STRAIN_STEP_SLOTS + fill++);
        ++P.rec.first.back();
        for (int k = 0; k < np_of(e); ++k) {
          const int v = vtx(e, k);
          if (stamp[v] != b) {
            stamp[v] = b;
            fstep[v] = st;
            touched.push_back(v);
          }
          lstep[v] = st;
        }
      }
    }
    // imports by group of first use; places reused once their vertex left in
    // a step whose group lies more than STRAIN_AHEAD groups back
    const int ngrp = (nstep + STRAIN_GROUP - 1) / STRAIN_GROUP;
    bystep.assign((size_t)ngrp, {});
    for (int32_t v : touched) bystep[fstep[v] / STRAIN_GROUP].push_back(v);
    std::vector<std::vector<int32_t>> leave((size_t)ngrp);
    std::vector<int32_t> freep;
    int used = 0;
    std::vector<uint8_t> lo_set((size_t)nband, 0), up_set((size_t)nband, 0);
    for (int g = 0; g < ngrp; ++g) {
      if (g - STRAIN_AHEAD - 1 >= 0)
        for (int32_t p : leave[g - STRAIN_AHEAD - 1]) freep.push_back(p);
      const size_t s0 = step0 + (size_t)g * STRAIN_GROUP;
      StrainGroup G{(int32_t)P.imp.size(), 0, -1, -1, P.rec.first[s0],
                    P.rec.first[std::min(s0 + STRAIN_GROUP, step0 + nstep)]};
      for (int32_t v : bystep[g]) {
        int p;
        if (!freep.empty()) {
          p = freep.back();
          freep.pop_back();
        } else {
          p = used++;
        }
        place[v] = p;
        leave[lstep[v] / STRAIN_GROUP].push_back(p);
        P.imp.push_back(StrainImport{(uint32_t)v, (uint32_t)p});
        if (pband[v] >= 0) {
          G.need_same = std::max(G.need_same, plevel[v]);
          lo_set[pband[v]] = 1;
        } else {
          G.need_prev = std::max(G.need_prev, vlast[v]);
          up_set[vband[v]] = 1;
        }
      }
      G.imp1 = (int32_t)P.imp.size();
      P.grp.push_back(G);
    }
    if (used > STRAIN_LDS_VERTS) return false;
    P.cap = std::max(P.cap, used);
    // records
    P.rec.packed.resize((size_t)P.rec.first.back());
    for (int32_t e : order) {
      StrainRec& r = P.rec.packed[(size_t)P.rec.at((size_t)P.slot[e])];
      r.np = (uint16_t)np_of(e);
      for (int k = 0; k < 3; ++k) {
        r.L0[k] = len0[4 * (size_t)e + k];
        r.place[k] = (uint16_t)place[vtx(e, k < r.np ? k : 0)];
      }
    }
    // exports by last step
    std::stable_sort(touched.begin(), touched.end(),
                     [&](int32_t a, int32_t c) { return lstep[a] < lstep[c]; });
    for (int32_t v : touched) {
      StrainExport x;
      x.v = (uint32_t)v;
      x.place = (uint32_t)place[v] | (vband[v] == b ? 0x80000000u : 0u);
      x.step = lstep[v];
      x.pad = 0;
      P.exp.push_back(x);
      pband[v] = b;
      plevel[v] = lvl_of_step[lstep[v]];
    }
    P.step_level.insert(P.step_level.end(), lvl_of_step.begin(), lvl_of_step.end());
    P.step_ptr.push_back((int32_t)(step0 + nstep));
    P.grp_ptr.push_back(P.grp_ptr.back() + ngrp);
    P.exp_ptr.push_back((int32_t)P.exp.size());
    for (int c = 0; c < nband; ++c) {
      if (lo_set[c]) P.lo.push_back(c);
      if (up_set[c]) P.up.push_back(c);
    }
    P.lo_ptr.push_back((int32_t)P.lo.size());
    P.up_ptr.push_back((int32_t)P.up.size());
  }
  P.rec.packed.resize(P.rec.packed.size() + STRAIN_STEP_SLOTS, StrainRec{});
  P.step_level.resize(P.step_level.size() + 64, std::numeric_limits<int32_t>::max());
  P.exp.resize(P.exp.size() + 64, StrainExport{0, 0, std::numeric_limits<int32_t>::max(), 0});
  P.lo.resize(P.lo.size() + 64, 0);
  P.up.resize(P.up.size() + 64, 0);
  return true;
}

}  // namespace cs
