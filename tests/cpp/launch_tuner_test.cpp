// The launch-shape tuner's choices from made-up pass times (cs_tune.h).
#include <algorithm>
#include <cstdio>

#include "../../collision_amd/csrc/cs_tune.h"

using namespace cs;

// Eight steps: a whole stream whose time per pair depends on the candidate
// (256 lanes fastest) and `inc` incremental passes of the other form, whose time per
// pair does not, as many more of them in the steps that run 256 lanes.
static int narrow_choice(int inc, bool inc_tuned) {
  LaunchTuner t(5000000, 256);
  int tr, na, qu;
  for (bool last = false; !last;) {
    t.candidates(&tr, &na, &qu);
    std::vector<TunePass> p;
    p.push_back({false, true, 1.0, na == 64 ? 1.3 : na == 128 ? 1.2 : 1.0, 1000000});
    for (int i = 0; i < (na == 256 ? 4 * inc : inc); ++i) p.push_back({true, inc_tuned, 0.1, 0.05, 3000});
    last = t.add_step(p);
  }
  t.choice(&tr, &na, &qu);
  return na;
}

int main() {
  LaunchTuner none(5000000, 256);
  int tr, na, qu;
  for (int i = 0; i < TUNE_STEPS; ++i) none.add_step({});
  none.choice(&tr, &na, &qu);
  if (tr != TUNE_TRAV_DEFAULT || na != TUNE_NARROW_DEFAULT || qu != TUNE_QUERY_DEFAULT) return 1;
  if (narrow_choice(0, false) != 256) return 2;
  // passes of the form that the candidate does not reach do not decide it
  if (narrow_choice(20, false) != 256) return 3;
  // (counted, they would)
  if (narrow_choice(20, true) == 256) return 4;
  // only candidates that launch differently are tried, and the default is among them
  const int CUS = 256, edge = 8 * CUS * 4 * 256;
  for (int n : {1, 4096, 32768, 32769, edge, edge + 1, 2 * edge + 1, 4 * edge + 1, 1 << 27}) {
    LaunchTuner t(n, CUS);
    std::vector<int> walks, queries;
    for (int i = 0; i < TUNE_STEPS; ++i) {
      t.candidates(&tr, &na, &qu);
      walks.push_back(traverse_grid(n, CUS, tr));
      queries.push_back(query_grid(n, qu));
      t.add_step({{false, true, 1.0, 1.0, 10}, {true, false, 1.0, 1.0, 10}});
    }
    auto count = [](std::vector<int> v) {
      std::sort(v.begin(), v.end());
      return (int)(std::unique(v.begin(), v.end()) - v.begin());
    };
    auto grids = [&](const int* cand, auto grid) {
      std::vector<int> v;
      for (int i = 0; i < 4; ++i) v.push_back(grid(cand[i]));
      return count(v);
    };
    const int gw = grids(TUNE_TRAV, [&](int c) { return traverse_grid(n, CUS, c); });
    const int gq = grids(TUNE_QUERY, [&](int c) { return query_grid(n, c); });
    if (gw != count(walks) || gq != count(queries)) return 5;
    // as many rounds of each as there are steps for: none shows up more often
    for (int i = 0; i < TUNE_STEPS; ++i)
      if ((walks[i] != walks[(i + gw) % TUNE_STEPS] && i + gw < TUNE_STEPS) ||
          (queries[i] != queries[(i + gq) % TUNE_STEPS] && i + gq < TUNE_STEPS))
        return 6;
    t.choice(&tr, &na, &qu);
    if (gw == 1 && tr != TUNE_TRAV_DEFAULT) return 7;
    if (gq == 1 && qu != TUNE_QUERY_DEFAULT) return 8;
  }
  std::puts("ok");
  return 0;
}
