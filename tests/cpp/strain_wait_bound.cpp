// How long a task of the banded strain sweep may have to wait, against the
// bound after which the kernel gives a wait up (strain_wait_us).
//
//   strain_wait_bound ring|fan|grid n
//
// A step may begin one step after the one before it, when the imports of its
// group are there; a task's progress and its waits are those of the kernel, all
// tasks run at once and everything else takes no time.  Prints the steps of a
// sweep, the longest wait of any import in steps and the bound in steps of 2 us.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../collision_amd/csrc/cs_strain_plan.h"

using namespace cs;

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  const int n = atoi(argv[2]);
  std::vector<int> ev;
  int nv = n;
  auto add = [&](int a, int b, int c) { ev.insert(ev.end(), {a, b, c, 0}); };
  if (!std::strcmp(argv[1], "ring")) {  // a closed string: vertex 0's visits are the first and the last
    for (int i = 0; i < n; ++i) add(i, (i + 1) % n, -1);
  } else if (!std::strcmp(argv[1], "fan")) {  // the hub is in every triangle
    nv = n + 2;
    for (int i = 0; i < n; ++i) add(0, i + 1, i + 2);
  } else {  // row-major sheet
    nv = n * n;
    for (int r = 0; r + 1 < n; ++r)
      for (int c = 0; c + 1 < n; ++c) {
        const int a = r * n + c;
        add(a, a + 1, a + n);
        add(a + 1, a + n + 1, a + n);
      }
  }
  const int ne = (int)(ev.size() / 4);
  std::vector<uint8_t> rigid((size_t)ne, 0);
  std::vector<double> len0(4 * (size_t)ne, 1.0);
  std::vector<int> lev;
  const int nl = strain_levels(nv, ne, ev.data(), rigid.data(), lev);
  StrainPlan P;
  if (!strain_build_plan(nv, ne, ev.data(), rigid.data(), len0.data(), lev, nl,
                         strain_band_count(ne, nl), P))
    return 3;
  const int K = 10, nb = P.nband;
  // done[step]: when the sweep before (or, for bands below, this one) finished it
  std::vector<int64_t> before(P.steps(), 0), now(P.steps(), 0);
  // when band b of a sweep has passed `level`: its last step at most there
  auto passed = [&](const std::vector<int64_t>& t, int b, int level) -> int64_t {
    const int32_t* l = P.step_level.data();
    const int s0 = P.step_ptr[b], s1 = P.step_ptr[b + 1];
    const int s = (int)(std::upper_bound(l + s0, l + s1, level) - l);
    return s > s0 ? t[s - 1] : 0;
  };
  int64_t longest = 0;
  for (int k = 0; k < K; ++k) {
    for (int b = 0; b < nb; ++b) {
      int64_t t = 0;
      for (int s = P.step_ptr[b], g = P.grp_ptr[b]; s < P.step_ptr[b + 1]; ++s) {
        if ((s - P.step_ptr[b]) % STRAIN_GROUP == 0) {
          const StrainGroup& G = P.grp[g++];
          int64_t ready = 0;
          if (G.need_same >= 0)
            for (int i = P.lo_ptr[b]; i < P.lo_ptr[b + 1]; ++i)
              ready = std::max(ready, passed(now, P.lo[i], G.need_same));
          if (k > 0 && G.need_prev >= 0)
            for (int i = P.up_ptr[b]; i < P.up_ptr[b + 1]; ++i)
              ready = std::max(ready, passed(before, P.up[i], G.need_prev));
          longest = std::max(longest, ready - t);
          t = std::max(t, ready);
        }
        now[s] = ++t;
      }
    }
    before = now;
  }
  std::printf("%zu %lld %lld\n", P.steps(), (long long)longest,
              (long long)(strain_wait_us((int64_t)P.steps(), K) / 2));
  return 0;
}
