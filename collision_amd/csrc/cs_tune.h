// The launch-shape tuner's candidates and scores (plain C++).  Over the first
// TUNE_STEPS steps every step runs one candidate of each launch shape; the
// kernel times are averaged per candidate and the fastest kept.
#pragma once
#include <algorithm>
#include <cstdint>
#include <vector>

namespace cs {

constexpr int TUNE_TRAV[4] = {4, 8, 16, 32};
constexpr int TUNE_NARROW[3] = {64, 128, 256};
constexpr int TUNE_QUERY[4] = {1024, 2048, 4096, 8192};
constexpr int TUNE_STEPS = 8;  // two rounds of the four-candidate lists
constexpr int TUNE_TRAV_DEFAULT = 8, TUNE_NARROW_DEFAULT = 128, TUNE_QUERY_DEFAULT = 4096;

// The full traversal's walks (cs_bvh.hip): each of the n leaves' walks in
// 2^traverse_cuts(n) parts, one per lane, on at most 8 x trav work-groups per CU.
constexpr int TRAV_THREADS = 256;
constexpr int TRAV_LANES = 262144, TRAV_SUB_MAX = 6;
inline int traverse_cuts(int n) {
  int lsub = 0;
  while (lsub < TRAV_SUB_MAX && ((int64_t)n << (lsub + 1)) <= TRAV_LANES) ++lsub;
  return lsub;
}
inline int traverse_grid(int n, int cus, int trav) {
  const int64_t need = (((int64_t)n << traverse_cuts(n)) + TRAV_THREADS - 1) / TRAV_THREADS;
  return (int)std::min<int64_t>(need, 8ll * cus * trav);
}
// the dirty query's wavefronts over the 2 n - 1 nodes
inline int query_grid(int n, int query) {
  return (int)std::min<int64_t>((2ll * n - 1 + 63) / 64, query);
}

// The candidates of a launch whose grids differ: of those with one grid the
// default, or else the first.  (A mesh that needs fewer work-groups than the smallest
// candidate allows launches the same for all of them: up to 2.1e6 elements for the
// traversal, 32,768 for the query.)
template <typename Grid>
inline std::vector<int> tune_distinct(const int* cand, int m, int def, Grid grid) {
  std::vector<int> out;
  for (int i = 0; i < m; ++i) {
    size_t j = 0;
    while (j < out.size() && grid(out[j]) != grid(cand[i])) ++j;
    if (j == out.size()) out.push_back(cand[i]);
    else if (cand[i] == def) out[j] = def;
  }
  return out;
}

// what a pass of a tuning step ran
struct TunePass {
  bool incremental;   // the dirty query ran, not the full traversal
  bool narrow_tuned;  // its narrow launches have the candidate's work-group size
  double ms_walk, ms_narrow;
  int64_t pairs;      // tested by the narrow phase
};

class LaunchTuner {
 public:
  // n elements on a device of `cus` compute units
  LaunchTuner(int n, int cus)
      : trav_{tune_distinct(TUNE_TRAV, 4, TUNE_TRAV_DEFAULT,
                            [&](int t) { return traverse_grid(n, cus, t); })},
        narrow_{{TUNE_NARROW, TUNE_NARROW + 3}},
        query_{tune_distinct(TUNE_QUERY, 4, TUNE_QUERY_DEFAULT,
                             [&](int q) { return query_grid(n, q); })} {}
  void candidates(int* trav, int* narrow, int* query) const {
    *trav = trav_.at(step_);
    *narrow = narrow_.at(step_);
    *query = query_.at(step_);
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
    trav_.add(step_, walk);
    query_.add(step_, query);
    narrow_.add(step_, narrow);
    return ++step_ >= TUNE_STEPS;
  }
  // the fastest of each (the default where nothing was measured)
  void choice(int* trav, int* narrow, int* query) const {
    *trav = trav_.best(TUNE_TRAV_DEFAULT);
    *narrow = narrow_.best(TUNE_NARROW_DEFAULT);
    *query = query_.best(TUNE_QUERY_DEFAULT);
  }
  int step() const { return step_; }

 private:
  struct Score {
    double ms = 0.0;
    int64_t n = 0;
  };
  struct Shape {
    std::vector<int> cand;
    std::vector<Score> score = std::vector<Score>(cand.size());
    int at(int step) const { return cand[(size_t)step % cand.size()]; }
    void add(int step, const Score& s) {
      if (!s.n) return;
      Score& to = score[(size_t)step % cand.size()];
      to.ms += s.ms / (double)s.n;
      to.n++;
    }
    int best(int def) const {
      int bi = -1;
      for (int i = 0; i < (int)cand.size(); ++i)
        if (score[i].n && (bi < 0 || score[i].ms / (double)score[i].n <
                                         score[bi].ms / (double)score[bi].n))
          bi = i;
      return bi < 0 ? def : cand[bi];
    }
  };
  int step_ = 0;
  Shape trav_, narrow_, query_;
};

}  // namespace cs
