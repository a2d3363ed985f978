// Launch shapes of the gather-GEMM: which output tile and how many K splits a
// product of given sizes takes.  Host code without state, kept apart from the
// kernels so that the rules can be tested without a GPU.
#pragma once

#include <algorithm>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"

namespace tn {
namespace kern {

constexpr int BK = 16;         // depth of a K tile
constexpr int kSkRanks = 512;  // stream-K grid: two workgroups per CU
constexpr int kMaxTileRows = 65535;  // workgroups of a launch in y (rows of tiles)

struct Plan {
  int BM, BN, splits, kps;
  bool sk = false;  // stream-K (128 x 128 tiles, kSkRanks workgroups)
};

// Stream-K layout of an M x N x K product on 128 x 128 tiles: whole rounds
// of kSkRanks tiles run data-parallel, the K iterations of the remaining
// tiles are split over the kSkRanks ranks.  Used when the remainder is at
// least half a round (below that a split tile has more than ~4 shares; the
// classic grid of two workgroups per CU leaves some CUs with one tile and
// others with two) and K is long enough (>= 64 iterations) for the shares to
// amortise their partial tiles.
struct SkLayout {
  int dp = 0, tiles = 0, nk = 0, S = 0;
  int64_t iters = 0;
  size_t part_bytes = 0, bytes = 0;
};
inline bool sk_layout(int M, int N, int K, SkLayout &L) {
  if (M < 128 || N < 128 || K <= 0) return false;
  const int64_t ntiles = (int64_t)ceil_div(M, 128) * ceil_div(N, 128);
  const int nk = ceil_div(K, BK);
  const int64_t dp = (ntiles / kSkRanks) * kSkRanks;
  const int64_t rest = ntiles - dp;
  if (rest < kSkRanks / 2 || nk < 64 || ntiles > (1 << 20)) return false;
  L.dp = (int)dp;
  L.tiles = (int)rest;
  L.nk = nk;
  L.iters = rest * nk;
  const int64_t lmax = ceil_div(L.iters, (int64_t)kSkRanks);
  L.S = (int)ceil_div(lmax, (int64_t)nk) + 1;
  L.part_bytes = (size_t)kSkRanks * L.S * 64 * 256 * sizeof(double);
  L.bytes = L.part_bytes + (size_t)L.tiles * sizeof(int);
  return true;
}

inline Plan choose(int M, int N, int K, bool f64) {
  Plan p;
  if (K <= 0) {
    p.BM = p.BN = 64;
    p.splits = 1;
    p.kps = 0;
    return p;
  }
  // Large outputs with a long K: 128 x 128 tiles.  (160 x 160 tiles would
  // fill the 256 CUs in one round at 2500 x 2500, but measured 1.03 ms
  // against 0.78 ms: their 25 accumulator tiles per wave leave too few
  // registers.)  With K of at most 8 tiles the 64 x 64 grid, four times the
  // workgroups at twice the occupancy, hides more of the short main loop's
  // prologue and epilogue: 2500 x 2500 x 100 in 47 us against 53 us.
  const int64_t tiles128 = (int64_t)ceil_div(M, 128) * ceil_div(N, 128);
  p.BM = p.BN = (M >= 128 && N >= 128 && tiles128 >= 200 && K > 8 * BK) ? 128 : 64;
  // 32 x 32 tiles (FP64) where the call is a few short workgroups: a K tile
  // takes 0.34 us in such a workgroup and 0.92 us in a 64 x 64 one (four times
  // the MFMAs per wave), so up to K = 400 the product needs no split, which
  // saves the reduction and its launch, and outputs of at most 32 rows or
  // columns waste less of the tile.  Back to back, with the host's 8.4 us per
  // call as the floor: 2500 x 128 x 128 13.2 to 8.1 us, 333 x 128 x 333 12.0
  // to 9.7, 1024 x 1024 x 64 10.4 to 8.4.  Above 2048 tiles the 64 x 64 grid
  // fills the chip and moves less through L2.  (A thin output of more than
  // 65535 rows of 32 tiles is past the grid's limit.)
  const int64_t tiles32 = (int64_t)ceil_div(M, 32) * ceil_div(N, 32);
  const bool thin = M <= 32 || N <= 32;
  if (f64 && K <= 400 && (thin || tiles32 <= 2048) && ceil_div(M, 32) <= kMaxTileRows) {
    p.BM = p.BN = 32;
    p.splits = 1;
    p.kps = ceil_div(K, BK) * BK;
    return p;
  }
  if (f64 && M <= 32 && N <= 32 && K >= 64 * 8 * BK) p.BM = p.BN = 32;
  const int64_t tiles = (int64_t)ceil_div(M, p.BM) * ceil_div(N, p.BN);
  // Split K when the tile grid cannot fill the 256 CUs and K is long: the
  // split count s that minimises the rounds of 256 workgroups per unit of
  // K work, ceil(tiles s / 256) / s, among those giving at least two
  // workgroups per CU (64 x 64 tiles run up to four per CU; one alone
  // leaves the MFMA pipe idle at every barrier), at least four K tiles per
  // split, fewest splits on a tie.  2500 x 128 x 2500 (80 tiles): 16 splits,
  // 51.5 us against 64.5 us at the 4 that merely reach 256 workgroups.
  p.splits = 1;
  if (tiles < 8 && K >= 64 * 8 * BK) {
    // a few tiles and a very long K (density matrices and their gradients,
    // 32 x 16 x 131072): the operands stream from HBM once, so as many
    // workgroups as 1024 over the tiles, at least eight K tiles each; 64
    // splits left three quarters of the CUs idle (133 to 143 us by layout,
    // 20 us now, the reduction included)
    p.splits = std::min(K / (8 * BK), 1024 / (int)tiles);
  } else if (tiles < 128 && K >= 4 * BK * 2) {
    const int maxs = std::max(1, K / (4 * BK));
    double best = 1e30;
    for (int sp = 1; sp <= std::min(maxs, 64); ++sp) {
      const int64_t wg = tiles * sp;
      if (wg < 512 && sp < maxs && sp < 64) continue;
      const double cost = (double)ceil_div(wg, (int64_t)256) / sp;
      if (cost < best - 1e-12) {
        best = cost;
        p.splits = sp;
      }
    }
  }
  p.kps = ceil_div(K, p.splits);
  p.kps = ceil_div(p.kps, BK) * BK;
  p.splits = ceil_div(K, p.kps);
  // stream-K only on request (GemmPlan{128, 0}): at 2500 x 2500 x 2500 it
  // measured 0.82 ms against 0.74 ms for the data-parallel grid
  return p;
}

// The heuristic plan, or the given launch shape with its K range rounded
// to whole tiles (at most one split per K tile).
inline Plan plan_for(int M, int N, int K, const GemmPlan *gp, bool f64) {
  if (gp == nullptr || gp->bm == 0 || K <= 0) return choose(M, N, K, f64);
  Plan p;
  p.BM = p.BN = gp->bm == 128 ? 128 : gp->bm == 32 && f64 ? 32 : 64;
  SkLayout L;
  if (p.BM == 128 && gp->splits == 0 && sk_layout(M, N, K, L)) {
    p.splits = 1;
    p.kps = ceil_div(K, BK) * BK;
    p.sk = true;
    return p;
  }
  const int maxs = std::max(1, ceil_div(K, BK));
  p.splits = std::min(std::max(gp->splits, 1), maxs);
  p.kps = ceil_div(ceil_div(K, p.splits), BK) * BK;
  p.splits = ceil_div(K, p.kps);
  return p;
}

// Launch shapes worth timing, the heuristic's own first; then the shapes
// around the heuristic of the 64 and 128 tiles, which every arithmetic has
// (in FP64 the heuristic's own may be a 32 tile without splits, around which
// no split count of the larger tiles would be tried).
inline std::vector<GemmPlan> candidates(int M, int N, int K, bool f64) {
  std::vector<GemmPlan> out;
  const Plan h = choose(M, N, K, f64), w = choose(M, N, K, false);
  auto add = [&](int bm, int splits) {
    if (bm == 128 && (M < 128 || N < 128)) return;
    GemmPlan g{bm, splits};
    const Plan r = plan_for(M, N, K, &g, f64);
    for (const auto &o : out) {
      const Plan e = plan_for(M, N, K, &o, f64);
      if (e.BM == r.BM && e.splits == r.splits && e.sk == r.sk) return;
    }
    out.push_back(g);
  };
  SkLayout L;
  add(h.BM, h.splits);
  add(w.BM, w.splits);
  add(64, 1);
  add(128, 1);
  if (sk_layout(M, N, K, L)) add(128, 0);  // splits 0 with bm 128: stream-K
  if (K >= 8 * BK) {
    add(64, std::max(2, w.splits * 2));
    add(64, std::max(2, w.splits / 2));
    add(128, std::max(2, w.splits));
  }
  return out;
}

}  // namespace kern
}  // namespace tn
