// The order of singular values: descending by rank_key, equal keys by index.
// A NaN gets the lowest key, so it comes after every number and the keys are
// totally ordered: the ranks of any p values are a permutation of 0..p-1.
// (Every comparison with NaN is false: ranks counted on the values themselves
// would repeat, and the permutation that gathers the singular vectors would
// keep unwritten entries.)
#pragma once

#include <limits>

namespace tn {

constexpr double rank_key(double v) {
  return v == v ? v : -std::numeric_limits<double>::infinity();
}

// whether the value of key u at index k comes before that of key v at index j
constexpr bool ranks_before(double u, int k, double v, int j) {
  return u > v || (u == v && k < j);
}

}  // namespace tn
