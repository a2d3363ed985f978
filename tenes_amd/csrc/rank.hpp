// The order of singular values: descending, NaN after every number, equal
// ones by index.  A total order, so the ranks of any p values are a
// permutation of 0..p-1 (every comparison with NaN is false: ranks counted
// with > and == alone would repeat, and the permutation that gathers the
// singular vectors would keep unwritten entries).
#pragma once

namespace tn {

// whether value u at index k comes before value v at index j
constexpr bool ranks_before(double u, int k, double v, int j) {
  const bool un = u != u, vn = v != v;
  if (un || vn) return un == vn ? k < j : vn;
  return u > v || (u == v && k < j);
}

}  // namespace tn
