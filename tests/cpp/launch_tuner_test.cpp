// The launch-shape tuner's choices from made-up pass times (cs_tune.h).
#include <cstdio>

#include "../../collision_amd/csrc/cs_tune.h"

using namespace cs;

// Eight steps: a whole stream whose time per pair depends on the candidate
// (256 lanes fastest) and `inc` incremental passes of the other form, whose time per
// pair does not, as many more of them in the steps that run 256 lanes.
static int narrow_choice(int inc, bool inc_tuned) {
  LaunchTuner t;
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
  LaunchTuner none;
  int tr, na, qu;
  for (int i = 0; i < TUNE_STEPS; ++i) none.add_step({});
  none.choice(&tr, &na, &qu);
  if (tr != TUNE_TRAV_DEFAULT || na != TUNE_NARROW_DEFAULT || qu != TUNE_QUERY_DEFAULT) return 1;
  if (narrow_choice(0, false) != 256) return 2;
  // passes of the form that the candidate does not reach do not decide it
  if (narrow_choice(20, false) != 256) return 3;
  // (counted, they would)
  if (narrow_choice(20, true) == 256) return 4;
  std::puts("ok");
  return 0;
}
