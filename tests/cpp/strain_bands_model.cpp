// CPU model of the banded strain-limit sweep (collision_amd/csrc/cs_strain_plan.h)
// against the sequential sweep loop (dcollid.cpp:486-596).
//
//   strain_bands_model topo.bin xnoise vnoise max_sweeps nband resident seed mistake
//
// The tasks (sweep, band) are started in order, at most `resident` at a time,
// and their three activities (imports of one group, one step, exports of the
// steps done) are interleaved at random, each only when the waits the device
// kernel makes are satisfied.  A task's window holds the imported values; a
// place that is read before its import or after its export is caught.
// mistake: 0 none, 1 imports do not wait for the previous sweep, 2 imports do
// not wait for the lower band, 3 places reused without waiting for the
// exports, 4 the visit of an unchanged vertex counts as changed only when the
// stamp is later than the step (a write in the previous sweep is forgotten).
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../collision_amd/csrc/cs_strain_plan.h"

using namespace cs;

struct Vec { double c[3]; };
static double dt = 1e-3;

static bool over(const Vec& o0, const Vec& o1, const Vec& a0, const Vec& a1, double len0, bool* deg) {
  double so = 0, sn = 0;
  for (int i = 0; i < 3; ++i) {
    const double d = o0.c[i] - o1.c[i];
    so += d * d;
    const double e = (o0.c[i] + dt * a0.c[i]) - (o1.c[i] + dt * a1.c[i]);
    sn += e * e;
  }
  const double lo = std::sqrt(so), ln = std::sqrt(sn);
  *deg = false;
  if (lo > 1e-10 && ln > 1e-10)
    return std::fabs((ln - len0) / len0) > 0.1 || std::fabs((ln - lo) / lo) > 0.1;
  *deg = true;
  return true;
}

struct Elem {
  int np;
  const Vec* x[3];
  Vec* a[3];
  const double* L0;
};
static int visit(Elem& s, uint32_t* wmask, int* degen) {
  int edges = 0;
  *wmask = 0;
  for (int k = 0; k < (s.np == 3 ? 3 : 1); ++k) {
    const int i = k, j = (k + 1) % 3;
    bool g;
    if (!over(*s.x[i], *s.x[j], *s.a[i], *s.a[j], s.L0[k], &g)) continue;
    for (int c = 0; c < 3; ++c) {
      const double m = 0.5 * (s.a[i]->c[c] + s.a[j]->c[c]);
      s.a[i]->c[c] = m;
      s.a[j]->c[c] = m;
    }
    *wmask |= (1u << i) | (1u << j);
    ++edges;
    if (g) ++*degen;
  }
  return edges;
}

int main(int argc, char** argv) {
  if (argc < 9) return 2;
  FILE* f = std::fopen(argv[1], "rb");
  const double xn = atof(argv[2]), vn = atof(argv[3]);
  const int max_sweeps = atoi(argv[4]);
  int nband = atoi(argv[5]);
  const int resident = atoi(argv[6]), seed = atoi(argv[7]), mistake = atoi(argv[8]);
  int nv, ne;
  if (!f || std::fread(&nv, 4, 1, f) != 1 || std::fread(&ne, 4, 1, f) != 1) return 2;
  std::vector<int> e3(3 * (size_t)ne), rg((size_t)ne);
  std::vector<Vec> x((size_t)nv), v((size_t)nv);
  std::vector<double> l3(3 * (size_t)ne);
  if (std::fread(e3.data(), 4, e3.size(), f) != e3.size() || std::fread(rg.data(), 4, rg.size(), f) != rg.size() ||
      std::fread(x.data(), 24, x.size(), f) != x.size() || std::fread(l3.data(), 8, l3.size(), f) != l3.size())
    return 2;
  std::fclose(f);
  std::mt19937_64 rng((uint64_t)seed);
  std::normal_distribution<double> N(0.0, 1.0);
  for (auto& p : x)
    for (double& c : p.c) c += xn * N(rng);
  for (auto& p : v)
    for (double& c : p.c) c = vn * N(rng);
  std::vector<int> ev(4 * (size_t)ne);
  std::vector<uint8_t> rigid((size_t)ne);
  std::vector<double> len0(4 * (size_t)ne, 0.0);
  for (int e = 0; e < ne; ++e) {
    for (int k = 0; k < 3; ++k) {
      ev[4 * (size_t)e + k] = e3[3 * (size_t)e + k];
      len0[4 * (size_t)e + k] = l3[3 * (size_t)e + k];
    }
    rigid[e] = (uint8_t)rg[e];
  }
  // the sequential loop
  std::vector<Vec> ref = v;
  int ref_sweeps = 0, ref_edges = 0, ref_degen = 0;
  for (int it = 0; it < max_sweeps; ++it) {
    int edges = 0;
    for (int e = 0; e < ne; ++e) {
      if (rigid[e]) continue;
      const int np = ev[4 * (size_t)e + 2] >= 0 ? 3 : 2;
      Elem s{np, {}, {}, &len0[4 * (size_t)e]};
      for (int k = 0; k < np; ++k) {
        s.x[k] = &x[ev[4 * (size_t)e + k]];
        s.a[k] = &ref[ev[4 * (size_t)e + k]];
      }
      uint32_t wm;
      edges += visit(s, &wm, &ref_degen);
    }
    ++ref_sweeps;
    ref_edges = edges;
    if (edges == 0) break;
  }
  // the banded sweeps
  std::vector<int> lev;
  const int nl = strain_levels(nv, ne, ev.data(), rigid.data(), lev);
  int64_t ns = 0;
  for (int e = 0; e < ne; ++e) ns += !rigid[e];
  if (nband <= 0) nband = strain_band_count(ns, nl);
  StrainPlan P;
  if (!strain_build_plan(nv, ne, ev.data(), rigid.data(), len0.data(), lev, nl, nband, P)) {
    std::printf("plan does not fit\n");
    return 3;
  }
  std::vector<Vec> av = v;
  std::vector<int64_t> stamp((size_t)nv, 0);
  int sweeps = 0, edges_last = 0, degen = 0;
  long long evals = 0, caught = 0;
  for (int k0 = 0; k0 < max_sweeps;) {
    const int K = std::min(10, max_sweeps - k0);
    std::vector<uint8_t> pre(P.rec.size(), 0);
    bool any = false;
    for (int e = 0; e < ne; ++e) {
      if (rigid[e]) continue;
      const int np = ev[4 * (size_t)e + 2] >= 0 ? 3 : 2;
      bool g, o = false;
      for (int k = 0; k < (np == 3 ? 3 : 1); ++k) {
        const int i = ev[4 * (size_t)e + k], j = ev[4 * (size_t)e + (k + 1) % 3];
        o = o || over(x[i], x[j], av[i], av[j], len0[4 * (size_t)e + k], &g);
      }
      pre[P.slot[e]] = o;
      any = any || o;
    }
    if (!any) {
      ++sweeps;
      edges_last = 0;
      break;
    }
    struct Task {
      int k, b, step = 0, done = 0, pos;
      int imp[STRAIN_IMPORT_WAVES];  // next group of each import wavefront
      std::vector<Vec> vel, xo;
      std::vector<int64_t> st;
      std::vector<int> owner;  // vertex held by a place, -1 none
      bool over = false;
    };
    const int nb = P.nband, ntask = K * nb;
    std::vector<int> prog((size_t)ntask), edges((size_t)K, 0);
    for (int i = 0; i < ntask; ++i) prog[i] = P.step_level[P.step_ptr[i % nb]] - 1;
    std::vector<Task> live;
    int next = 0, finished = 0;
    auto min_prog = [&](const std::vector<int32_t>& p, const std::vector<int32_t>& l, int b, int k) {
      int m = INT32_MAX;
      for (int i = p[b]; i < p[b + 1]; ++i) m = std::min(m, prog[(size_t)k * nb + l[i]]);
      return m;
    };
    long idle = 0;
    while (finished < ntask) {
      while (next < ntask && (int)live.size() < resident) {
        Task t;
        t.k = next / nb;
        t.b = next % nb;
        for (int i = 0; i < STRAIN_IMPORT_WAVES; ++i) t.imp[i] = i;
        t.pos = P.exp_ptr[t.b];
        t.vel.resize((size_t)P.cap);
        t.xo.resize((size_t)P.cap);
        t.st.assign((size_t)P.cap, 0);
        t.owner.assign((size_t)P.cap, -1);
        live.push_back(t);
        ++next;
      }
      Task& t = live[rng() % live.size()];
      const int what = (int)(rng() % (2 + STRAIN_IMPORT_WAVES)) - STRAIN_IMPORT_WAVES;
      const int nstep = P.step_ptr[t.b + 1] - P.step_ptr[t.b], ngrp = P.grp_ptr[t.b + 1] - P.grp_ptr[t.b];
      bool moved = false;
      if (what < 0) {  // one group of imports
        int& next_g = t.imp[what + STRAIN_IMPORT_WAVES];
        const int g = next_g;
        bool ok = g < ngrp;
        const StrainGroup G = ok ? P.grp[(size_t)P.grp_ptr[t.b] + g] : StrainGroup{};
        if (ok && mistake != 3) ok = t.done >= STRAIN_GROUP * (g - STRAIN_AHEAD);
        if (ok && mistake != 2 && G.need_same >= 0)
          ok = min_prog(P.lo_ptr, P.lo, t.b, t.k) >= G.need_same;
        if (ok && mistake != 1 && t.k > 0 && G.need_prev >= 0)
          ok = min_prog(P.up_ptr, P.up, t.b, t.k - 1) >= G.need_prev;
        if (ok) {
          for (int i = G.imp0; i < G.imp1; ++i) {
            const uint32_t u = P.imp[i].v, p = P.imp[i].place;
            if (t.owner[p] >= 0) ++caught;  // still in use
            t.owner[p] = (int)u;
            t.vel[p] = av[u];
            t.xo[p] = x[u];
            t.st[p] = stamp[u];
          }
          next_g += STRAIN_IMPORT_WAVES;
          moved = true;
        }
      } else if (what == 0) {  // one step
        const int g = t.step / STRAIN_GROUP;
        if (t.step < nstep && t.imp[g % STRAIN_IMPORT_WAVES] > g) {
          const size_t s = (size_t)P.step_ptr[t.b] + t.step;
          const int64_t L = P.step_level[s], nl64 = P.n_levels;
          const int64_t thr = t.k > 0 ? 1 + (t.k - 1) * nl64 + L + (mistake == 4 ? 1 : 0) : 1;
          for (int i = 0; i < STRAIN_STEP_SLOTS; ++i) {
            const StrainRec& r = P.rec[s * STRAIN_STEP_SLOTS + i];
            if (!r.np) continue;
            bool act = t.k == 0 && pre[s * STRAIN_STEP_SLOTS + i];
            for (int q = 0; q < r.np; ++q) {
              if (t.owner[r.place[q]] < 0) ++caught;  // not imported
              act = act || t.st[r.place[q]] >= thr;
            }
            if (!act) continue;
            ++evals;
            Elem el{r.np, {}, {}, r.L0};
            for (int q = 0; q < r.np; ++q) {
              el.x[q] = &t.xo[r.place[q]];
              el.a[q] = &t.vel[r.place[q]];
            }
            uint32_t wm;
            edges[t.k] += visit(el, &wm, &degen);
            for (int q = 0; q < r.np; ++q)
              if ((wm >> q) & 1u) t.st[r.place[q]] = 1 + t.k * nl64 + L;
          }
          ++t.step;
          moved = true;
        }
      } else if (t.step > t.done) {  // exports of the steps done
        const int n = t.step;
        for (; t.pos < P.exp_ptr[t.b + 1] && P.exp[t.pos].step < n; ++t.pos) {
          const StrainExport& q = P.exp[t.pos];
          const int p = (int)(q.place & 0x7fffffffu);
          if (t.owner[p] != (int)q.v) ++caught;
          av[q.v] = t.vel[p];
          stamp[q.v] = (q.place >> 31) && t.k == K - 1 ? 0 : t.st[p];
          t.owner[p] = -1;
        }
        t.done = n;
        prog[(size_t)t.k * nb + t.b] =
            n < nstep ? P.step_level[(size_t)P.step_ptr[t.b] + n] - 1 : INT32_MAX;
        moved = true;
        if (n == nstep) {
          if (t.pos != P.exp_ptr[t.b + 1]) ++caught;
          ++finished;
          live.erase(live.begin() + (&t - live.data()));
        }
      }
      idle = moved ? 0 : idle + 1;
      if (idle > 400000) {
        std::printf("deadlock: %d of %d tasks done\n", finished, ntask);
        return 4;
      }
    }
    int nz = 0;
    while (nz < K && edges[nz] > 0) ++nz;
    sweeps += nz < K ? nz + 1 : K;
    edges_last = nz < K ? 0 : edges[K - 1];
    k0 += K;
    if (nz < K) break;
  }
  long long differ = 0, left = 0;
  for (int i = 0; i < nv; ++i) {
    if (std::memcmp(&av[i], &ref[i], sizeof(Vec)) != 0) ++differ;
    left += stamp[i] != 0;
  }
  std::printf("bands=%d levels=%d steps=%zu window=%d sweeps=%d/%d edges=%d/%d degenerate=%d/%d evals=%lld\n",
              P.nband, nl, P.steps(), P.cap, sweeps, ref_sweeps, edges_last, ref_edges, degen, ref_degen, evals);
  std::printf("vertices differing=%lld misuse=%lld stamps left=%lld\n", differ, caught, left);
  return differ || caught || left || sweeps != ref_sweeps || edges_last != ref_edges || degen != ref_degen;
}
