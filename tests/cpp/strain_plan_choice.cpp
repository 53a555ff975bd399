// Which strain sweep a sheet's element order gets: prints whether a plan fits,
// whether it pays, its imports per vertex and its window in bytes.
//
//   strain_plan_choice n rows|cols|radial|random|tiles<k>|within<k>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <random>

#include "../../collision_amd/csrc/cs_strain_plan.h"

using namespace cs;

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  const int n = atoi(argv[1]), nv = n * n;
  const char* kind = argv[2];
  std::vector<int> tri;
  for (int r = 0; r + 1 < n; ++r)
    for (int c = 0; c + 1 < n; ++c) {
      const int a = r * n + c;
      tri.insert(tri.end(), {a, a + 1, a + n, a + 1, a + n + 1, a + n});
    }
  const int ne = (int)tri.size() / 3;
  std::mt19937 g(3);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  std::vector<double> key((size_t)ne);
  std::vector<double> tile;
  const int k = std::strpbrk(kind, "0123456789") ? atoi(std::strpbrk(kind, "0123456789")) : 1;
  for (int e = 0; e < ne; ++e) {
    const double row = e / 2 / (n - 1), col = e / 2 % (n - 1);
    if (!std::strncmp(kind, "rows", 4)) key[e] = e;
    else if (!std::strncmp(kind, "cols", 4)) key[e] = col * n + row;
    else if (!std::strncmp(kind, "radial", 6)) key[e] = std::hypot(row - n / 2, col - n / 2);
    else if (!std::strncmp(kind, "random", 6)) key[e] = U(g);
    else if (!std::strncmp(kind, "within", 6)) key[e] = e + k * U(g);
    else {
      if ((size_t)(e / k) == tile.size()) tile.push_back(U(g));
      key[e] = tile[e / k];
    }
  }
  std::vector<int> p((size_t)ne), ev;
  std::iota(p.begin(), p.end(), 0);
  std::stable_sort(p.begin(), p.end(), [&](int a, int b) { return key[a] < key[b]; });
  for (int e : p) ev.insert(ev.end(), {tri[3 * e], tri[3 * e + 1], tri[3 * e + 2], 0});
  std::vector<uint8_t> rigid((size_t)ne, 0);
  std::vector<double> len0(4 * (size_t)ne, 1.0);
  std::vector<int> lev;
  const int nl = strain_levels(nv, ne, ev.data(), rigid.data(), lev);
  StrainPlan P;
  int nb = strain_band_count(ne, nl);
  bool fits;
  while (!(fits = strain_build_plan(nv, ne, ev.data(), rigid.data(), len0.data(), lev, nl, nb, P)) &&
         nb < STRAIN_MAX_BANDS)
    nb = std::min(2 * nb, STRAIN_MAX_BANDS);
  std::printf("%d %d %.3f %d\n", fits, fits && strain_plan_pays(P),
              fits ? (double)P.imp.size() / (double)nv : 0.0, P.cap * STRAIN_VERT_BYTES);
  return 0;
}
