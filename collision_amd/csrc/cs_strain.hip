// Banded strain-limit sweeps: reduceSuperelast (dcollid.cpp:486-596) by one
// work-group per (sweep, band of the element order), velocities in LDS.
//
// The plan (cs_strain_plan.h) explains bands, levels, steps, imports and
// exports, and why the tasks cannot deadlock when they are started in the
// order (sweep, band): every task takes its number from a counter, so the
// lowest unfinished one is always resident and only waits for lower ones.
//
// What bounds it: the chain of steps.  An element's result feeds the next
// level, so a sweep is `levels` dependent steps (4,090 on a 1024 x 1024 cloth)
// however many compute units take part; the sweeps and bands follow each other
// a few steps apart.  A step is one wavefront's work on LDS only (three stamp
// reads; where an element has to be evaluated, its vertices and the edges'
// tests), and everything that touches memory is done by the task's other
// wavefronts ahead of it or behind it:
//   wavefront 0     steps
//   wavefronts 1,2  imports: wait for the other tasks' progress, load the
//                   vertices of a group of steps into LDS (alternate groups)
//   wavefront 3     exports and the task's published progress
//
// Kernel time per time step, against all sweeps in one work-group (k_strain_pipe,
// whose level iterations each scanned ten rows of marks, loaded 256 B records
// and crossed two barriers): 64 x 64 cloth, every edge over the limit, 1.76 ->
// 0.39 ms; 256 x 256 17.0 -> 1.15 ms (1.3e6 evaluations, 0.95 us a step, of which
// 0.76 us evaluation); 1024 x 1024 cloth with 2,000 strings, few edges over the
// limit, 8.2 -> 2.7 ms (0.17-0.37 us a step); 64 scenes 1.5 -> 0.52 ms.  The
// pre-check replaces a packing and a check kernel (0.58 -> below 0.06 ms at 1024^2).
//
// An element is evaluated in sweep k only if its result can differ from
// "nothing over the limit": a vertex of it was written since its visit in
// sweep k - 1, by it or by another element (for the first sweep of a launch:
// since the launch began, or the pre-check found an edge over the limit).
// Every vertex carries the stamp 1 + sweep * levels + level of its last write
// (0: none in this launch) in the fourth component of avgVel; the last visit of
// the last sweep stores 0 again.
//
// Values cross work-groups (and XCDs, each with its own L2) as relaxed
// agent-scope accesses, which go to the device's coherence point; the progress
// of a task is stored after all stores of its exports have been acknowledged.
// No agent-scope fence is needed (it would write back and invalidate L2).
#include <algorithm>

#include "cs_internal.h"
#include "cs_strain_edge.h"

namespace cs {

namespace {

constexpr int SB_IMPORT = STRAIN_IMPORT_WAVES;
constexpr int SB_THREADS = 64 * (2 + SB_IMPORT);
constexpr int SB_POLLS = 256;  // polls of a wait between looks at the clock and the abort flags

// words of DevState::bands.stat
enum { SBS_TICKET = 0, SBS_DONE = 1, SBS_EDGES = 2, SBS_DEGEN = 2 + SB_MAX_SWEEPS, SBS_EVALS, SBS_ABORT };
static_assert(SBS_ABORT < SB_STAT_INTS, "stat words");

// A vertex of the window: avgVel, the stamp of its last write, x_old.  Seven
// 8-byte words, an odd count, so that lanes reading different places spread
// over the LDS banks (64 B records put all of them on a quarter).
struct BandVertex {
  double v[3];
  int stamp, pad;
  double x[3];
};
static_assert(sizeof(BandVertex) == STRAIN_VERT_BYTES, "BandVertex layout");

__device__ inline unsigned long long agent_load(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void agent_store(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline int lds_load(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// LDS flags between the task's wavefronts: a wavefront's LDS accesses are
// executed in order, so the flag is written after the data before it and what
// is read after the flag is current; only the compiler has to keep the order.
__device__ inline void lds_order() { asm volatile("" ::: "memory"); }
__device__ inline void lds_publish(int* p, int v) {
  lds_order();
  if ((threadIdx.x & 63) == 0) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The bookkeeping of one wait: false when it must be given up, because another
// wait was or because it has lasted longer than all steps of the launch could
// take one after another (strain_wait_us; only an inconsistent plan does).  It
// is measured in time, not in polls: a wait in LDS polls some ten times faster
// than one in memory.  Time between two looks counts up to B.look_ticks, so
// that a wavefront that was not running meanwhile does not run out of it.
struct Spin {
  int n = 0;
  long long last = 0, ticks = 0;
  __device__ inline bool go(const int* s_abort, const StrainBands& B) {
    if (++n < SB_POLLS) return true;
    n = 0;
    if (lds_load(s_abort)) return false;
    if (__hip_atomic_load(B.stat + SBS_ABORT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
    const long long now = (long long)wall_clock64();
    if (last) ticks += min(now - last, B.look_ticks);
    last = now;
    if (ticks >= B.wait_ticks) {
      if ((threadIdx.x & 63) == 0)
        __hip_atomic_store(B.stat + SBS_ABORT, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    return true;
  }
};

static_assert(STRAIN_TOL == CS_SUPERELAS_TOL && STRAIN_MIN_LEN == CS_ROUND_EPS, "cs_strain_edge.h");

__device__ inline double sq_f64(const double* a, const double* b) {
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const double d = a[i] - b[i];
    s += d * d;
  }
  return s;
}
__device__ inline void end_position(const double* o, const double* a, double dt, double* p) {
#pragma unroll
  for (int i = 0; i < 3; ++i) p[i] = o[i] + dt * a[i];
}

}  // namespace

// Pre-check with the velocities at the start of the launch, in element order
// (neighbouring elements share the gathered vertices): the byte of every
// element's slot, and the any-edge flag.  Also resets the tasks' progress and
// statistics.  count: the elements over the limit are counted (CNT_STRAIN_OVER).
__global__ void __launch_bounds__(256)
    k_strain_precheck(const int4* __restrict__ ev, const dvec4* __restrict__ len0,
                      const int32_t* __restrict__ slot, const dvec4* __restrict__ x_old,
                      const dvec4* __restrict__ av, double dt, int ne, uint8_t* __restrict__ pre,
                      int* __restrict__ prog, int ntask, int nband,
                      const int32_t* __restrict__ step_ptr, const int32_t* __restrict__ step_level,
                      int* __restrict__ stat, int* __restrict__ counters, int count) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  // (a task has nothing to do below its band's first level)
  for (int i = e; i < ntask; i += gridDim.x * blockDim.x)
    prog[(size_t)i * SB_PROG_STRIDE] = step_level[step_ptr[i % nband]] - 1;
  if (e < SB_STAT_INTS) stat[e] = 0;
  if (counters[CNT_STRAIN_FLAG] < 0) return;  // loop already finished
  bool any = false;
  if (e < ne) {
    const int s = slot[e];
    if (s >= 0) {
      const int4 t = ev[e];
      const dvec4 L = len0[e];
      const double len[3] = {L.x, L.y, L.z};
      double o[3][3], p[3][3];
      const int vid[3] = {t.x, t.y, t.z >= 0 ? t.z : t.x};
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const dvec4 x = x_old[vid[i]], v = av[vid[i]];
        const double a[3] = {v.x, v.y, v.z};
        o[i][0] = x.x; o[i][1] = x.y; o[i][2] = x.z;
        end_position(o[i], a, dt, p[i]);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        if (i > 0 && t.z < 0) break;
        const int j = (i + 1) % 3;
        const double so = sq_f64(o[i], o[j]), sn = sq_f64(p[i], p[j]);
        int r = edge_screen(sn, edge_limits(so, len[i]));
        if (r < 0) r = edge_exact(so, sn, len[i]);
        any = any || r > 0;
      }
      pre[s] = any ? 1 : 0;
    }
  }
  const uint64_t over = __ballot(any);
  if (over && (threadIdx.x & 63) == 0) {
    atomicOr(&counters[CNT_STRAIN_FLAG], 1);
    if (count) atomicAdd(&counters[CNT_STRAIN_OVER], __popcll(over));
  }
}

static void launch_precheck(hipStream_t st, DevState& S, double dt, int count) {
  const StrainBands& B = S.bands;
  hipLaunchKernelGGL(k_strain_precheck, dim3((S.ne + 255) / 256), dim3(256), 0, st, S.ev, S.len0,
                     B.slot, S.x_old, S.av, dt, S.ne, B.pre, B.prog, SB_MAX_SWEEPS * B.nband,
                     B.nband, B.step_ptr, B.step_level, B.stat, S.counters, count);
}
void launch_strain_count(hipStream_t st, DevState& S, double dt) { launch_precheck(st, S, dt, 1); }

__global__ void __launch_bounds__(SB_THREADS)
    k_strain_bands(StrainBands B, const dvec4* __restrict__ x_old, dvec4* av, double dt, int K,
                   int* __restrict__ counters) {
  extern __shared__ __align__(64) unsigned char s_raw[];
  BandVertex* win = reinterpret_cast<BandVertex*>(s_raw);  // the task's window
  __shared__ int s_task, s_flag, s_step, s_done, s_imp[SB_IMPORT], s_abort;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid == 0) {
    s_flag = counters[CNT_STRAIN_FLAG];  // <0 finished, 0 no edge over the limit, >0 sweeps needed
    s_task = s_flag < 0 ? 0 : atomicAdd(B.stat + SBS_TICKET, 1);
    s_step = s_done = s_abort = 0;
    for (int i = 0; i < SB_IMPORT; ++i) s_imp[i] = i;  // next group of each
  }
  __syncthreads();
  if (s_flag < 0) return;
  const int nb = B.nband, task = __builtin_amdgcn_readfirstlane(s_task), k = task / nb, b = task - k * nb;
  if (s_flag == 0) {  // nothing over the limit: this sweep is a no-op and ends the loop
    // (a work-group that starts late may read the -1 instead: it returns too)
    if (task == 0 && tid == 0) {
      counters[CNT_STRAIN_FLAG] = -1;
      counters[CNT_STRAIN_EDGES] = 0;
      atomicAdd(&counters[CNT_STRAIN_SWEEPS], 1);
    }
    return;
  }
  const int step0 = B.step_ptr[b], nstep = B.step_ptr[b + 1] - step0;
  const int NL = B.n_levels;
  int* stat = B.stat;
  if (wave == 0) {
    // --- the steps.  Records (static) are loaded one group ahead into
    // registers.  The lanes past the step's last element hold the records of the
    // steps after it, or the unused ones at the end, and take no part.  (Holding them
    // to the last record is slower: 96 x 96 drape 324 -> 335 us a launch.)
    static_assert(STRAIN_GROUP == 4, "unrolled by hand");
    const int32_t* row_ptr = B.row_ptr + step0;
    StrainRec r[4];
    int pr[4], n[4];
    // step u's records and pre-check bytes: [row, end), none past the last step
    auto load = [&](int u, int row, int end) {
      n[u] = end - row;
      r[u] = (B.rec + row)[lane];
      pr[u] = k == 0 ? (B.pre + row)[lane] : 0;
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) load(u, row_ptr[min(u, nstep)], row_ptr[min(u + 1, nstep)]);
    // of the 64 steps from s on: levels; first records a group later, and one more
    int lv = B.step_level[step0 + min(lane, nstep)];
    int rw = row_ptr[min(4 + lane, nstep)], rw1 = row_ptr[min(5 + lane, nstep)];
    int edges = 0, degen = 0, evals = 0;
    bool ok = true;
    for (int s = 0; s < nstep && ok; s += 4) {
      const int g = s >> 2;
      if ((s & 63) == 0 && s > 0) {
        lv = B.step_level[step0 + min(s + lane, nstep)];
        rw = row_ptr[min(s + 4 + lane, nstep)];
        rw1 = row_ptr[min(s + 5 + lane, nstep)];
      }
      for (Spin sp; lds_load(&s_imp[g % SB_IMPORT]) <= g;) {
        if (!sp.go(&s_abort, B)) {
          ok = false;
          break;
        }
      }
      if (!ok) break;
      lds_order();
      // the stamps of all four steps, read again once a step has written
      int t[4][3];
      auto stamps = [&](int u) {
#pragma unroll
        for (int i = 0; i < 3; ++i) t[u][i] = win[r[u].place[i]].stamp;
      };
#pragma unroll
      for (int u = 0; u < 4; ++u) stamps(u);
      bool wrote = false;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int L = __builtin_amdgcn_readlane(lv, (s + u) & 63);
        const int thr = k > 0 ? 1 + (k - 1) * NL + L : 1;
        if (wrote) stamps(u);
        // (place[2] of a bond repeats place[0])
        const StrainRec q = r[u];
        // (no short circuit: the stamp reads would be put off behind it)
        const bool act = (lane < n[u]) & ((pr[u] != 0) | (t[u][0] >= thr) | (t[u][1] >= thr) | (t[u][2] >= thr));
        // the same step of the next group
        load(u, __builtin_amdgcn_readlane(rw, (s + u) & 63), __builtin_amdgcn_readlane(rw1, (s + u) & 63));
        if (__ballot(act)) {
          if (act) {
            BandVertex* w[3] = {win + q.place[0], win + q.place[1], win + q.place[2]};
            double a[3][3], o[3][3], p[3][3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
#pragma unroll
              for (int c = 0; c < 3; ++c) {
                a[i][c] = w[i]->v[c];
                o[i][c] = w[i]->x[c];
              }
              end_position(o[i], a[i], dt, p[i]);
            }
            EdgeLimits lim[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) lim[i] = edge_limits(sq_f64(o[i], o[(i + 1) % 3]), q.L0[i]);
            uint32_t wm = 0u;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              const int j = (i + 1) % 3;
              const double sn = sq_f64(p[i], p[j]);
              int v = edge_screen(sn, lim[i]);
              if (i > 0 && q.np != 3) v = 0;
              if (v < 0) v = edge_exact(sq_f64(o[i], o[j]), sn, q.L0[i]);
              if (v > 0) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                  double vt = a[i][c] + a[j][c];
                  vt = 0.5 * vt;
                  a[i][c] = vt;
                  a[j][c] = vt;
                }
                end_position(o[i], a[i], dt, p[i]);
                end_position(o[j], a[j], dt, p[j]);
                wm |= (1u << i) | (1u << j);
                ++edges;
                degen += v >> 1;
              }
            }
            const int st = 1 + k * NL + L;
#pragma unroll
            for (int i = 0; i < 3; ++i)
              if ((wm >> i) & 1u) {
#pragma unroll
                for (int c = 0; c < 3; ++c) w[i]->v[c] = a[i][c];
                w[i]->stamp = st;
              }
            ++evals;
          }
          wrote = true;
          lds_publish(&s_step, min(s + u + 1, nstep));
        }
      }
      lds_publish(&s_step, min(s + 4, nstep));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      edges += __shfl_xor(edges, o);
      degen += __shfl_xor(degen, o);
      evals += __shfl_xor(evals, o);
    }
    if (lane == 0) {
      if (edges) atomicAdd(stat + SBS_EDGES + k, edges);
      if (degen) atomicAdd(stat + SBS_DEGEN, degen);
      if (evals) atomicAdd(stat + SBS_EVALS, evals);
    }
    if (!ok) lds_publish(&s_abort, 1);
  } else if (wave <= SB_IMPORT) {
    // --- imports, every SB_IMPORT-th group
    const int grp0 = B.grp_ptr[b], ngrp = B.grp_ptr[b + 1] - grp0;
    const int nlo = B.lo_ptr[b + 1] - B.lo_ptr[b], nup = B.up_ptr[b + 1] - B.up_ptr[b];
    const int lob = lane < nlo ? B.lo[B.lo_ptr[b] + lane] : -1;
    const int upb = lane < nup ? B.up[B.up_ptr[b] + lane] : -1;
    // wait until the listed bands' tasks of sweep `row` have reached `need`
    auto wait_for = [&](int nbr, int row, int need, int& seen) -> bool {
      if (seen >= need) return true;
      const int* p = B.prog + ((size_t)row * nb + (nbr < 0 ? 0 : nbr)) * SB_PROG_STRIDE;
      for (Spin sp;;) {
        int v = INT32_MAX;
        if (nbr >= 0) v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__ballot(v < need) == 0) {
#pragma unroll
          for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
          seen = v;
          return true;
        }
        if (!sp.go(&s_abort, B)) return false;
        __builtin_amdgcn_s_sleep(1);
      }
    };
    int seen_lo = -1, seen_up = -1;
    bool ok = true;
    // The entries of a group are loaded while the group before it is
    // fetched, their x_old (constant) before the waits.
    StrainImport e[2] = {};
    StrainGroup G{0, 0, -1, -1, 0, 0}, Gn = G;
    if (wave - 1 < ngrp) {
      G = B.grp[grp0 + wave - 1];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (G.imp0 + 64 * j + lane < G.imp1) e[j] = B.imp[G.imp0 + 64 * j + lane];
    }
    for (int g = wave - 1; g < ngrp; g += SB_IMPORT) {
      dvec4 xo[2];
      bool has[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        has[j] = G.imp0 + 64 * j + lane < G.imp1;
        if (has[j]) xo[j] = x_old[e[j].v];
      }
      if (g + SB_IMPORT < ngrp) Gn = B.grp[grp0 + g + SB_IMPORT];
      else Gn.imp0 = Gn.imp1 = 0;
      uint32_t warm = 0u, warmp = 0u;
      {  // bring the group's records (up to 64 lines of 128 B) and pre-check bytes into L2
        const int n = G.rec1 - G.rec0;
        if (4 * lane < n) warm = *reinterpret_cast<const uint32_t*>(B.rec + G.rec0 + 4 * lane);
        if (k == 0 && STRAIN_STEP_SLOTS * lane < n) warmp = B.pre[G.rec0 + STRAIN_STEP_SLOTS * lane];
      }
      // places of vertices that left more than STRAIN_AHEAD groups ago
      for (Spin sp; lds_load(&s_done) < STRAIN_GROUP * (g - STRAIN_AHEAD);) {
        if (!sp.go(&s_abort, B)) {
          ok = false;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      if (ok && G.need_same >= 0) ok = wait_for(lob, k, G.need_same, seen_lo);
      if (ok && k > 0 && G.need_prev >= 0) ok = wait_for(upb, k - 1, G.need_prev, seen_up);
      if (!ok) break;
      asm volatile("" ::: "memory");
      auto put = [&](const StrainImport& im, const unsigned long long* q, const dvec4& x) {
        BandVertex& w = win[im.place];
        w.v[0] = __longlong_as_double((long long)q[0]);
        w.v[1] = __longlong_as_double((long long)q[1]);
        w.v[2] = __longlong_as_double((long long)q[2]);
        w.stamp = (int)q[3];
        w.x[0] = x.x;
        w.x[1] = x.y;
        w.x[2] = x.z;
      };
      unsigned long long q[2][4];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (has[j]) {
          const unsigned long long* p = reinterpret_cast<const unsigned long long*>(av + e[j].v);
#pragma unroll
          for (int c = 0; c < 4; ++c) q[j][c] = agent_load(p + c);
        }
      StrainImport en[2] = {};
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (Gn.imp0 + 64 * j + lane < Gn.imp1) en[j] = B.imp[Gn.imp0 + 64 * j + lane];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (has[j]) put(e[j], q[j], xo[j]);
      for (int i = G.imp0 + 128 + lane; i < G.imp1; i += 64) {
        const StrainImport im = B.imp[i];
        const unsigned long long* p = reinterpret_cast<const unsigned long long*>(av + im.v);
#pragma unroll
        for (int c = 0; c < 4; ++c) q[0][c] = agent_load(p + c);
        put(im, q[0], x_old[im.v]);
      }
      lds_publish(&s_imp[wave - 1], g + SB_IMPORT);
      asm volatile("" ::"v"(warm), "v"(warmp));
      G = Gn;
      e[0] = en[0];
      e[1] = en[1];
    }
    if (!ok) lds_publish(&s_abort, 1);
  } else {
    // --- exports, and the level below which this task is done
    int pos = B.exp_ptr[b];
    const int end = B.exp_ptr[b + 1];
    int* prog = B.prog + (size_t)task * SB_PROG_STRIDE;
    StrainExport e = B.exp[pos + lane];
    int lvbase = 0, lv = B.step_level[step0 + min(lane, nstep)];
    bool ok = true;
    for (int done = 0; done < nstep;) {
      int n = done;
      for (Spin sp; (n = lds_load(&s_step)) <= done;) {
        if (!sp.go(&s_abort, B)) {
          ok = false;
          break;
        }
      }
      if (!ok) break;
      lds_order();
      for (;;) {
        const bool mine = pos + lane < end && e.step < n;
        if (mine) {
          const BandVertex& w = win[e.place & 0x7fffffffu];
          unsigned long long* p = reinterpret_cast<unsigned long long*>(av + e.v);
          // (k_strain_bands leaves no stamp behind)
          const int st = (e.place >> 31) && k == K - 1 ? 0 : w.stamp;
          agent_store(p, (unsigned long long)__double_as_longlong(w.v[0]));
          agent_store(p + 1, (unsigned long long)__double_as_longlong(w.v[1]));
          agent_store(p + 2, (unsigned long long)__double_as_longlong(w.v[2]));
          agent_store(p + 3, (unsigned long long)(unsigned)st);
        }
        const int c = __popcll(__ballot(mine));
        pos += c;
        if (c) e = B.exp[pos + lane];
        if (c < 64) break;
      }
      lds_publish(&s_done, n);
      int level = INT32_MAX;
      if (n < nstep) {
        if (n - lvbase >= 64) {
          lvbase = n;
          lv = B.step_level[step0 + min(n + lane, nstep)];
        }
        level = __shfl(lv, n - lvbase) - 1;
      }
      // every export has been acknowledged before the progress is stored
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == 0) __hip_atomic_store(prog, level, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      done = n;
    }
    if (!ok) lds_publish(&s_abort, 1);
  }
  __syncthreads();
  if (tid == 0) {
    if (s_abort) atomicOr(&counters[CNT_ERR], CS_DEVERR_STRAIN);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the statistics' atomics
    if (atomicAdd(stat + SBS_DONE, 1) == K * nb - 1) {  // the last task
      auto get = [&](int i) {
        return __hip_atomic_load(stat + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      int nz = 0;
      while (nz < K && get(SBS_EDGES + nz) > 0) ++nz;
      const int niter = nz < K ? nz + 1 : K;  // sweeps the sequential loop runs
      counters[CNT_STRAIN_EDGES] = nz < K ? 0 : get(SBS_EDGES + K - 1);
      counters[CNT_STRAIN_DEGEN] += get(SBS_DEGEN);
      counters[CNT_STRAIN_SWEEPS] += niter;
      counters[CNT_STRAIN_LEVELS] += niter * NL;
      counters[CNT_STRAIN_EVALS] += get(SBS_EVALS);
      counters[CNT_STRAIN_FLAG] = (nz == K) ? 0 : -1;  // all K wrote: the loop goes on
    }
  }
}

hipError_t strain_bands_setup(DevState& S) {
  StrainBands& B = S.bands;
  int device = 0, khz = 0;
  CS_HIP_RET(hipGetDevice(&device));
  CS_HIP_RET(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device));
  B.wait_ticks = strain_wait_us(B.steps, SB_MAX_SWEEPS) * khz / 1000;
  B.look_ticks = 10ll * khz;  // 10 ms
  if ((size_t)S.bands.cap * sizeof(BandVertex) <= 65536) return hipSuccess;
  // (the same bound for every handle: a later, smaller one must not lower it)
  return hipFuncSetAttribute(reinterpret_cast<const void*>(k_strain_bands),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             STRAIN_LDS_VERTS * (int)sizeof(BandVertex));
}

hipError_t strain_limit_bands(hipStream_t st, DevState& S, double dt, int max_sweeps,
                              std::vector<hipEvent_t>* marks) {
  const StrainBands& B = S.bands;
  for (int k0 = 0; k0 < max_sweeps;) {
    const int K = std::min(SB_MAX_SWEEPS, max_sweeps - k0);
    launch_precheck(st, S, dt, 0);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (marks && hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess)
      (void)hipEventRecord(e0, st);
    hipLaunchKernelGGL(k_strain_bands, dim3(K * B.nband), dim3(SB_THREADS),
                       (size_t)B.cap * sizeof(BandVertex), st, B, S.x_old, S.av, dt, K, S.counters);
    if (e1) {
      (void)hipEventRecord(e1, st);
      marks->push_back(e0);
      marks->push_back(e1);
    }
    k0 += K;
  }
  return hipGetLastError();
}

}  // namespace cs
