// Bytes of the banded strain sweep's records for one string of n bonds, against
// the 256 bytes an element that the one-work-group sweep takes.
//
//   strain_plan_size n
#include <cstdio>
#include <cstdlib>

#include "../../collision_amd/csrc/cs_strain_plan.h"

using namespace cs;

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  const int n = atoi(argv[1]);
  std::vector<int> ev;
  for (int i = 0; i < n; ++i) ev.insert(ev.end(), {i, i + 1, -1, 0});
  std::vector<uint8_t> rigid((size_t)n, 0);
  std::vector<double> len0(4 * (size_t)n, 1.0);
  std::vector<int> lev;
  const int nl = strain_levels(n + 1, n, ev.data(), rigid.data(), lev);
  StrainPlan P;
  if (!strain_build_plan(n + 1, n, ev.data(), rigid.data(), len0.data(), lev, nl,
                         strain_band_count(n, nl), P))
    return 3;
  // every element has its record, read as a row of its step or packed
  for (int e = 0; e < n; ++e)
    if (P.rec[(size_t)P.slot[e]].np != 2 || P.rec[(size_t)P.slot[e]].L0[0] != 1.0) return 4;
  size_t used = 0;
  for (size_t i = 0; i < P.rec.size(); ++i) used += P.rec[i].np != 0;
  if (used != (size_t)n) return 5;
  std::printf("%zu %zu\n", P.rec.packed.size() * sizeof(StrainRec), (size_t)n * 256);
  return 0;
}
