// The launch-shape tuner's candidates and scores (plain C++).  Over the first
// TUNE_STEPS steps every step runs one candidate of each launch shape; the
// kernel times are averaged per candidate and the fastest kept.
#pragma once
#include <cstdint>
#include <vector>

namespace cs {

constexpr int TUNE_TRAV[4] = {4, 8, 16, 32};
constexpr int TUNE_NARROW[3] = {64, 128, 256};
constexpr int TUNE_QUERY[4] = {1024, 2048, 4096, 8192};
constexpr int TUNE_STEPS = 8;  // two rounds of the four-candidate lists
constexpr int TUNE_TRAV_DEFAULT = 8, TUNE_NARROW_DEFAULT = 128, TUNE_QUERY_DEFAULT = 4096;

// what a pass of a tuning step ran
struct TunePass {
  bool incremental;   // the dirty query ran, not the full traversal
  bool narrow_tuned;  // its narrow launches have the candidate's work-group size
  double ms_walk, ms_narrow;
  int64_t pairs;      // tested by the narrow phase
};

class LaunchTuner {
 public:
  void candidates(int* trav, int* narrow, int* query) const {
    *trav = TUNE_TRAV[step_ % 4];
    *narrow = TUNE_NARROW[step_ % 3];
    *query = TUNE_QUERY[step_ % 4];
  }
  // the passes of a step that ran candidates(); true when it was the last one
  bool add_step(const std::vector<TunePass>& passes) {
    Score walk, query, narrow;
    for (const TunePass& p : passes) {
      Score& s = p.incremental ? query : walk;
      s.ms += p.ms_walk;
      s.n++;
      if (!p.narrow_tuned) continue;
      narrow.ms += p.ms_narrow;
      narrow.n += p.pairs > 0 ? p.pairs : 0;
    }
    auto add = [](Score& to, const Score& s) {
      if (!s.n) return;
      to.ms += s.ms / (double)s.n;
      to.n++;
    };
    add(trav_[step_ % 4], walk);
    add(query_[step_ % 4], query);
    add(narrow_[step_ % 3], narrow);
    return ++step_ >= TUNE_STEPS;
  }
  // the fastest of each (the default where nothing was measured)
  void choice(int* trav, int* narrow, int* query) const {
    *trav = best(trav_, TUNE_TRAV, 4, TUNE_TRAV_DEFAULT);
    *narrow = best(narrow_, TUNE_NARROW, 3, TUNE_NARROW_DEFAULT);
    *query = best(query_, TUNE_QUERY, 4, TUNE_QUERY_DEFAULT);
  }
  int step() const { return step_; }

 private:
  struct Score {
    double ms = 0.0;
    int64_t n = 0;
  };
  static int best(const Score* s, const int* cand, int m, int def) {
    int bi = -1;
    for (int i = 0; i < m; ++i)
      if (s[i].n && (bi < 0 || s[i].ms / (double)s[i].n < s[bi].ms / (double)s[bi].n)) bi = i;
    return bi < 0 ? def : cand[bi];
  }
  int step_ = 0;
  Score trav_[4], narrow_[3], query_[4];
};

}  // namespace cs
