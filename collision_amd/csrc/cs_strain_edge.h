// One edge of reduceSuperelastOnce (dcollid.cpp:486-560): is it over the strain
// or the strain-rate limit.  Plain C++ for the host and the device.
#pragma once
#include <cmath>

#ifdef __HIPCC__
#define CS_EDGE_FN __host__ __device__ inline
#else
#define CS_EDGE_FN inline
#endif

namespace cs {

constexpr double STRAIN_TOL = 0.10;        // dcollid.cpp:489
constexpr double STRAIN_MIN_LEN = 1e-10;   // shorter edges are degenerate (collid.h:17)

// The test on squared lengths: with s the squared length at the end of the step,
// |sqrt(s) / l - 1| > 0.1 for the rest length or the x_old length l is a
// comparison of s with 1.1^2 l^2 and 0.9^2 l^2, without a square root or a
// division in the chain from edge to edge.  The exact test rounds a handful of
// times (each within 2^-53 relative), the limits here likewise, and a decision is
// taken only beyond 1e-9 from the limit, so it is the exact one.  All in FP64
// (ratios from FP32 reciprocals, certain to 1e-6, took the same time: 256 x 256
// cloth 1.17 ms a launch, 64 x 64 0.40).
// Inputs nearer to a limit, degenerate lengths, rest lengths that are not
// positive and anything not finite run the exact test.
struct EdgeLimits {
  double over_hi, over_lo, under_hi, under_lo;
  bool fine;
};
constexpr double STRAIN_MARGIN = 1e-9;
constexpr double STRAIN_MIN_SQ = 4e-20;  // (twice the degenerate length) squared

// so: squared x_old length
CS_EDGE_FN EdgeLimits edge_limits(double so, double len0) {
  constexpr double a = 1.0 + STRAIN_TOL + STRAIN_MARGIN, b = 1.0 - STRAIN_TOL - STRAIN_MARGIN;
  constexpr double c = 1.0 + STRAIN_TOL - STRAIN_MARGIN, d = 1.0 - STRAIN_TOL + STRAIN_MARGIN;
  const double s0 = len0 * fabs(len0);  // (not positive where len0 is not)
  // (fmin and fmax drop a NaN, the sum does not)
  const double lo = fmin(s0, so), hi = fmax(s0, so);
  const bool fine = (lo > 2.0 * STRAIN_MIN_SQ) & (s0 + so < 1e200);
  return EdgeLimits{a * a * lo, b * b * hi, c * c * lo, d * d * hi, fine};
}
// 1 over, 0 under, -1 not certain; s: squared length at the end positions (where
// the limits are fine the lower ones of "over" alone can meet a degenerate s)
CS_EDGE_FN int edge_screen(double s, const EdgeLimits& L) {
  const bool over = L.fine & ((s > L.over_hi) | ((s < L.over_lo) & (s > STRAIN_MIN_SQ)));
  const bool under = L.fine & (s < L.under_hi) & (s > L.under_lo);
  return (int)over - (int)!(over | under);  // (no branch)
}
// 0 under, 1 over, 3 over and degenerate
CS_EDGE_FN int edge_exact(double so, double s, double len0) {
  const double len_old = sqrt(so), len_new = sqrt(s);  // dist3 of the same points
  if (len_old > STRAIN_MIN_LEN && len_new > STRAIN_MIN_LEN) {
    const double strain_rate = (len_new - len_old) / len_old;
    const double strain = (len_new - len0) / len0;
    return (fabs(strain) > STRAIN_TOL || fabs(strain_rate) > STRAIN_TOL) ? 1 : 0;
  }
  return 3;
}

}  // namespace cs
