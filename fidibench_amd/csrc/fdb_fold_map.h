// fdb_fold_map.h -- the integer map of a run of additions inside one binade
// (see fdb_fold.hip), as the device kernel and the CPU test program of the
// host code both compile it.
#ifndef FDB_FOLD_MAP_H
#define FDB_FOLD_MAP_H

#include <hip/hip_runtime.h>

#include <cmath>

namespace fdb {

// Effect of a run of values on m: d[p] is added to an m of parity p; lo
// and hi bound the offsets from the starting m after each value (both
// parities; the trajectories of the two differ by at most 1).
struct FoldMap {
  double d0, d1, lo, hi;
};

__host__ __device__ inline FoldMap fold_identity() {
  return {0.0, 0.0, __builtin_inf(), -__builtin_inf()};
}

__host__ __device__ inline bool fold_odd(double d) {  // |d| < 2^53, an integer
  const double h = 0.5 * d;
  return h != floor(h);
}

// The run of a, then that of b.
__host__ __device__ inline FoldMap fold_then(const FoldMap& a, const FoldMap& b) {
  FoldMap r;
  r.d0 = a.d0 + (fold_odd(a.d0) ? b.d1 : b.d0);
  r.d1 = a.d1 + (fold_odd(a.d1) ? b.d0 : b.d1);  // start 1: parity 1 + d1
  r.lo = fmin(a.lo, fmin(a.d0, a.d1) + b.lo);
  r.hi = fmax(a.hi, fmax(a.d0, a.d1) + b.hi);
  return r;
}

// The run of m, then the one value v (in units of u, |v| < 2^52).  Split at
// trunc(v): v - trunc(v) is exact for every v, so only a tie compares equal
// to half a unit.  (v - floor(v) is not on (-0.5, 0): the value next to -0.5
// rounds to half a unit there.)
__host__ __device__ inline void fold_append(FoldMap& m, double v) {
  const double t = trunc(v), r = fabs(v - t), away = t + copysign(1.0, v);
  double d0 = r > 0.5 ? away : t, d1 = d0;
  if (r == 0.5) {  // to the even m
    d0 = fold_odd(m.d0 + t) ? away : t;
    d1 = fold_odd(m.d1 + t) ? t : away;
  }
  m.d0 += d0;
  m.d1 += d1;
  m.lo = fmin(m.lo, fmin(m.d0, m.d1));
  m.hi = fmax(m.hi, fmax(m.d0, m.d1));
}

// How far (in u) the loop's s may be from the sum in another order that
// guesses it: half a unit for each of the loop's n additions, which drift one
// way where all round alike (2^27 values of 0.1: a relative 2^-28.7), and the
// other sum's few.  (Where |s| was in a higher binade before, it may be
// further off: fold_step sees that.)
__host__ __device__ inline double fold_slack(unsigned long long n) {
  return 0.5 * (double)n + 16384.0;
}

// Whether s stays in its binade from the guessed start m0 on, through every
// value, however the slack falls.
__host__ __device__ inline bool fold_fits(double m0, double lo, double hi, double slack) {
  const double first = 4503599627370496.0 + slack, last = 2.0 * 4503599627370496.0 - slack;
  return m0 >= first && m0 <= last && m0 + lo >= first && m0 + hi <= last;
}

}  // namespace fdb

#endif
