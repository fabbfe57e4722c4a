// fps_rounds_bound.hpp -- how a threshold round's bound and step follow from the last round,
// usable in the kernels and on the host (the CPU test that checks the picks by it).
#pragma once
#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define FPSX_BOUND __host__ __device__ __forceinline__
#else
#define FPSX_BOUND inline
#endif

namespace fpsx {

// A point's key: (min-distance, index) in 64 bits, larger first; 0 is below every point.
FPSX_BOUND uint64_t make_key(int value_bits, uint32_t tie) {
  return ((uint64_t)((uint32_t)value_bits + 1u) << 32) | tie;
}

// The best key of a point at distance 0 from a pick, as every pick is from itself.
constexpr uint64_t kZeroKey = ((uint64_t)1 << 32) | 0xffffffffu;

// The bound of the next round, whose candidates are the points above it; no key exceeds T.
// A round's picks fall to keys of distance 0, where their index counts against the points that
// lay there before.  So as long as some point may lie above those keys, none of them is a
// candidate: the first pick among them comes from a round of its own, which sees all picks.
FPSX_BOUND uint64_t round_bound(uint64_t T, uint64_t step) {
  const uint64_t b = T > step ? T - step : 0;
  return T > kZeroKey && b < kZeroKey ? kZeroKey : b;
}

// The step after a round of C candidates: the square root damps it against the count's noise,
// and it at most doubles, since a round with too many candidates for the list takes one pick (2^20
// clustered points, 16384 picks: 205 rounds and 2118 us where it could grow fourfold and doubled
// after every round without candidates too, 196 and 2035 so).
FPSX_BOUND uint64_t next_step(uint64_t step, uint32_t target, uint32_t C) {
  double r = sqrt((double)target / (double)C);
  r = r > 2.0 ? 2.0 : r;
  const double ns = (double)step * r;
  return ns < 1.0 ? 1 : (ns > 4.0e18 ? (uint64_t)1 << 61 : (uint64_t)ns);
}

// The step after a round of C candidates that were too many.
FPSX_BOUND uint64_t less_step(uint64_t step, uint32_t target, uint32_t C) {
  const uint64_t ns = (uint64_t)((double)step * sqrt((double)target / (double)C));
  return ns < 1 ? 1 : ns;
}

}  // namespace fpsx
