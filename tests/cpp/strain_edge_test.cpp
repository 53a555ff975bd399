// The strain limit's screen (cs_strain_edge.h) against its exact test, over
// lengths of all sizes and end lengths at, near and far from every limit.
//   prints: cases, wrong decisions, certain cases left undecided
#include <cfloat>
#include <cstdio>
#include <random>
#include <vector>

#include "../../collision_amd/csrc/cs_strain_edge.h"

using namespace cs;

int main() {
  std::mt19937_64 g(7);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  const double rest[] = {0.0, -1.0, -0.0, 5e-324, 1e-160, 1e-140, 1e-12, 1e-10, 2e-10, 1e-3, 0.1, 1.0,
                         1e6, 1e99, 1e101, 1e200, DBL_MAX, HUGE_VAL, -HUGE_VAL, NAN};
  long long cases = 0, wrong = 0, open = 0;
  auto check = [&](double so, double s, double len0, bool certain) {
    ++cases;
    const int r = edge_screen(s, edge_limits(so, len0)), e = edge_exact(so, s, len0);
    if (r >= 0 && r != e) ++wrong;
    if (r < 0 && certain) ++open;
  };
  const double off[] = {0.0, 1e-16, 1e-12, 5e-10, 1e-9, 2e-9, 1e-8, 1e-6, 1e-4, 1e-2, 0.3};
  for (int it = 0; it < 20000; ++it) {
    // ordinary lengths: everything farther than 2e-9 from a limit must be decided
    const double l0 = std::exp(20.0 * (U(g) - 0.7)), lo = l0 * (0.7 + 0.6 * U(g));
    if (l0 < 1e-9 || lo < 1e-9) continue;
    for (double base : {l0, lo})
      for (double lim : {0.9, 1.1, 1.0})
        for (double d : off)
          for (int sign = -1; sign <= 1; sign += 2) {
            const double len = base * lim * (1.0 + sign * d);
            double near = HUGE_VAL;
            for (double b : {l0, lo})
              for (double m : {0.9, 1.1}) near = std::fmin(near, std::fabs(len / b - m));
            check(lo * lo, len * len, l0, near > 3e-9);
          }
  }
  // rest lengths and squares of every kind against each other
  std::vector<double> sq = {0.0, 5e-324, 1e-300, 1e-21, 1e-20, 3.9e-20, 4.1e-20, 1e-19, 1e-6, 0.81, 1.0, 1.21,
                            1e12, 1e199, 1e201, DBL_MAX, HUGE_VAL, NAN};
  for (double l0 : rest)
    for (double so : sq)
      for (double s : sq) check(so, s, l0, false);
  std::printf("%lld %lld %lld\n", cases, wrong, open);
  return 0;
}
