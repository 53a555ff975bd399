// Host time of the strain schedules of a shuffled n x n sheet, whose vertex
// windows fit at no band count, against the time of its levels alone.
//   prints: levels, failed plan and other schedule, in seconds (best of three)
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../collision_amd/csrc/cs_internal.h"

using namespace cs;

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  const int n = atoi(argv[1]), nv = n * n;
  std::vector<int4> ev;
  for (int r = 0; r + 1 < n; ++r)
    for (int c = 0; c + 1 < n; ++c) {
      const int a = r * n + c;
      ev.push_back(make_int4(a, a + 1, a + n, 0));
      ev.push_back(make_int4(a + 1, a + n + 1, a + n, 0));
    }
  std::shuffle(ev.begin(), ev.end(), std::mt19937(1));
  const int ne = (int)ev.size();
  const int* e4 = reinterpret_cast<const int*>(ev.data());
  std::vector<uint8_t> ef((size_t)ne, EF_TRI), rigid((size_t)ne, 0);
  std::vector<double> len0(4 * (size_t)ne, 1.0);
  double levels = 1e30, rest = 1e30;
  for (int rep = 0; rep < 3; ++rep) {
    auto now = [] { return std::chrono::steady_clock::now(); };
    auto seconds = [](auto a, auto b) { return std::chrono::duration<double>(b - a).count(); };
    std::vector<int> lev, level;
    const auto t0 = now();
    const int nl = strain_levels(nv, ne, e4, rigid.data(), lev);
    const auto t1 = now();
    StrainPlan P;
    int nb = strain_band_count(ne, nl);
    while (!strain_build_plan(nv, ne, e4, rigid.data(), len0.data(), lev, nl, nb, P) &&
           nb < STRAIN_MAX_BANDS)
      nb = std::min(2 * nb, STRAIN_MAX_BANDS);
    if (!P.exp_ptr.empty() && P.exp_ptr.size() == (size_t)nb + 1) return 3;  // it fits
    int levels2 = 0, delta = 0;
    build_strain_schedule(nv, ne, ev.data(), ef.data(), lev, nl, level, levels2, delta);
    const auto t2 = now();
    if (levels2 < nl) return 4;
    // every element above the earlier ones of its vertices
    std::vector<int> last((size_t)nv, -1);
    for (int e = 0; e < ne; ++e)
      for (int v : {ev[e].x, ev[e].y, ev[e].z}) {
        if (level[e] <= last[v]) return 5;
        last[v] = level[e];
      }
    levels = std::min(levels, seconds(t0, t1));
    rest = std::min(rest, seconds(t1, t2));
  }
  std::printf("%g %g\n", levels, rest);
  return 0;
}
