// FP64 dense linear algebra building blocks for the truncated-SVD projector.
//
//  * randn            : counter-based normal numbers for the range finder.
//  * chol_inv_upper   : shifted Cholesky G + shift I = R^T R and R^{-1}, one
//                       workgroup with the p x p matrix resident in LDS
//                       (p <= 128).  Used by shifted CholeskyQR; wider Gram
//                       matrices (p <= 256) are factorised as two blocks
//                       (chol_prep, chol_assemble).
//  * jacobi_svd       : one-sided (Hestenes) Jacobi SVD, one workgroup per
//                       matrix, the whole m x p matrix resident in LDS (in
//                       global memory above 128), the p/2 column pairs of a
//                       round-robin step processed by 64 groups of 16 lanes.  The (c, s) of every rotation
//                       is streamed to HBM so the accumulated right factor can
//                       be rebuilt row-parallel afterwards (jacobi_accumulate)
//                       without keeping a second p x p matrix in LDS.
//  * qrp              : row-pivoted QR, the preconditioner of the exact path's
//                       Jacobi (m, n <= 128).
//  * sort_desc        : rank sort of singular values, descending (rank.hpp).
#include <cfloat>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "kernels.hpp"
#include "rank.hpp"

namespace tn {
namespace kern {

namespace {

constexpr int kMaxDim = 128;
typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

__global__ void randn_kernel(double *p, int64_t n, uint64_t seed,
                             uint64_t counter) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    const uint64_t j = counter + (uint64_t)(i >> 1);
    const uint64_t h1 = splitmix64(seed ^ (2 * j));
    const uint64_t h2 = splitmix64(seed ^ (2 * j + 1));
    const double u1 = ((double)(h1 >> 11) + 1.0) * 0x1.0p-53;  // (0, 1]
    const double u2 = (double)(h2 >> 11) * 0x1.0p-53;          // [0, 1)
    const double r = sqrt(-2.0 * log(u1));
    const double th = 6.283185307179586476925286766559 * u2;
    p[i] = (i & 1) ? r * sin(th) : r * cos(th);
  }
}

// One workgroup per column j of the n x p row-major block X: a column whose
// entries are all zero, or whose singular value sigma[j] is at most
// rel * sigma[0] (sigma may be null), is refilled with normal numbers (same
// generator and element numbering as randn_kernel).
__global__ void refill_columns_kernel(double *X, int64_t n, int p,
                                      const double *sigma, double rel,
                                      uint64_t seed, uint64_t counter) {
  __shared__ double part[256];
  const int j = blockIdx.x;
  const bool null_dir = sigma != nullptr && !(sigma[j] > rel * sigma[0]);
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const double v = X[i * p + j];
    acc += v * v;
  }
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (part[0] != 0.0 && !null_dir) return;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const int64_t e = i * p + j;
    const uint64_t c = counter + (uint64_t)(e >> 1);
    const uint64_t h1 = splitmix64(seed ^ (2 * c));
    const uint64_t h2 = splitmix64(seed ^ (2 * c + 1));
    const double u1 = ((double)(h1 >> 11) + 1.0) * 0x1.0p-53;
    const double u2 = (double)(h2 >> 11) * 0x1.0p-53;
    const double r = sqrt(-2.0 * log(u1));
    const double th = 6.283185307179586476925286766559 * u2;
    X[e] = (e & 1) ? r * sin(th) : r * cos(th);
  }
}

// ---------------------------------------------------------------------------
// Shifted Cholesky + inverse of the upper factor: blocked, one workgroup of
// 8 waves, the padded matrix resident in LDS, diagonally scaled first.
//
// One CU and a chain of p dependent pivots bound it, so everything that is
// not on that chain runs beside it.  Blocks of 16.  The 16 x 16 diagonal
// block is factored by one wave with column lc in lane lc of each 16-lane row
// (the four rows do the same work), an element of another column coming by
// DPP row_newbcast: a pivot step is a broadcast, a reciprocal square root and
// one multiply before the next pivot is known.  Per block column kb, two
// phases:
//   A  block row of F (forward substitution, one thread per column, the
//      diagonal block's entries again by DPP) and, on another wave, the
//      inverse of the diagonal block;
//   B  wave 0 updates the next diagonal block and factors it while the other
//      waves do the rest of the trailing update on the FP64 MFMA.
// Alone on the device, average over a projector's calls at 128 x 128: 93 us
// before (4 waves, pivots through LDS with a division each, substitutions
// through LDS broadcasts, the inverse after the factor), 40 us now; 8 x 8:
// 14.8 us before, 5.6 us now.
// ---------------------------------------------------------------------------
constexpr int kCholThreads = 512;
constexpr int kCholWaves = kCholThreads / 64;
// row length of the LDS matrix: odd against bank conflicts, and one constant
// for every p so that the offsets are immediates
constexpr int kCholLd = kMaxDim + 1;
constexpr int kCholXdLd = 17;  // padded leading dimension of the diagonal inverses

__device__ __forceinline__ d4 mfma16(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Orders one wave's LDS accesses around an exchange between its own lanes:
// the stores before the fence are complete before the loads after it.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <class F, int... I>
__device__ __forceinline__ void unroll_impl(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unroll(F f) {
  unroll_impl(f, std::make_integer_sequence<int, N>{});
}

// v of lane L of the caller's 16-lane row (all lanes of the row active)
template <int L>
__device__ __forceinline__ double row_bcast(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x150 + L, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x150 + L, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// 1 / sqrt(x) for positive normal x: the hardware estimate and two Newton
// steps y += y (1/2 - (x/2) y^2).
__device__ __forceinline__ double rsqrt_newton(double x) {
  const double h = 0.5 * x;
  double y = __builtin_amdgcn_rsq(x);
#pragma unroll
  for (int i = 0; i < 2; ++i) y = fma(y, fma(-h * y, y, 0.5), y);
  return y;
}

size_t chol_lds_bytes(int p) {
  const int pp = (p + 15) / 16 * 16;
  return ((size_t)pp * kCholLd + (size_t)pp * kCholXdLd) * sizeof(double);
}

// FULL: p == kMaxDim (every pass of the range finder).
template <bool FULL>
__global__ __launch_bounds__(kCholThreads) void chol_inv_kernel(
    const double *G, int p_arg, double shift_coef, double rel_floor, double *R,
    double *Rinv, const double *pre) {
  extern __shared__ double lds[];
  __shared__ int defic[kMaxDim];
  __shared__ double s_diag[kMaxDim], s_dg[kMaxDim], s_scl[kMaxDim];
  __shared__ double s_rd[kMaxDim];  // 1 / F[i][i] (0 for a dropped column)
  __shared__ double s_shift, s_thr, s_floor;
  __shared__ int s_zero, s_near;
  const int p = FULL ? kMaxDim : p_arg;
  const int pp = (p + 15) / 16 * 16;  // padded size (identity padding)
  const int nb = pp / 16;
  constexpr int ld = kCholLd;
  // A: pp x ld, the upper triangle of 16 x 16 blocks holds G, then F; below
  // it block (bj, bi) holds the transpose of X's block (bi, bj), bi < bj
  double *A = lds;
  double *Xd = lds + (size_t)pp * ld;  // nb blocks of 16 x kCholXdLd: F_kk^-1
  const int tid = threadIdx.x;
  // the wave's number as a scalar: its branches are uniform
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane >> 4, lc = lane & 15;  // (row in 4-group, column)
  const int c0 = lane, r0 = w;               // load/store mapping

  // Load: thread -> columns c0, c0 + 64 and rows r0 + 8u.  The full size
  // holds its 32 values in registers (all loads in flight together) until the
  // scales are known; smaller ones go through LDS.
  double v[FULL ? 16 : 1][2];
  if (tid == 0) s_near = 1;
  if constexpr (FULL) {
#pragma unroll
    for (int u = 0; u < 16; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) v[u][h] = G[(r0 + 8 * u) * kMaxDim + c0 + 64 * h];
    if (tid < kMaxDim) s_diag[tid] = G[tid * (kMaxDim + 1)];
  } else {
    for (int r = r0; r < pp; r += kCholWaves)
      for (int c = c0; c < pp; c += 64) {
        const double g = r < p && c < p ? G[r * p + c] : (r == c ? 1.0 : 0.0);
        A[r * ld + c] = g;
        if (r == c) s_diag[r] = g;
      }
  }
  __syncthreads();
  // Diagonal (Jacobi) scaling G -> D G D, D = diag(G)^{-1/2}: the factor of
  // the scaled matrix is R~ with R = R~ D^{-1}, R^{-1} = D R~^{-1}.  Column
  // norms no longer enter the conditioning (a block of nearly orthogonal
  // columns of very different lengths factors as well as an orthonormal
  // one); zero columns keep a zero diagonal.
  // A pre-scaled input (pre != nullptr: a diagonal block or Schur
  // complement of a larger scaled and shifted Gram matrix) keeps unit scales.
  if (tid < pp) {
    const double g = s_diag[tid];
    const double dg = (tid < p && !pre) ? (g > 0.0 ? sqrt(g) : 0.0) : 1.0;
    s_dg[tid] = dg;
    s_scl[tid] = dg > 0.0 ? 1.0 / dg : 0.0;
  }
  __syncthreads();
  {
    bool near = true;
    if constexpr (FULL) {
      const double sc[2] = {s_scl[c0], s_scl[c0 + 64]};
#pragma unroll
      for (int u = 0; u < 16; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int r = r0 + 8 * u, c = c0 + 64 * h;
          const double g = (v[u][h] * s_scl[r]) * sc[h];
          A[r * ld + c] = g;
          near = near && fabs(g - (r == c ? 1.0 : 0.0)) <= 1e-10;
        }
    } else {
      for (int r = r0; r < pp; r += kCholWaves)
        for (int c = c0; c < pp; c += 64) {
          const double g = (A[r * ld + c] * s_scl[r]) * s_scl[c];
          A[r * ld + c] = g;
          near = near && fabs(g - (r == c ? 1.0 : 0.0)) <= 1e-10;
        }
    }
    if (!near) s_near = 0;
  }
  if (w == 0) {
    double tr = 0.0, mx = 0.0;
    for (int i = lane; i < p; i += 64) {
      const double g = (s_diag[i] * s_scl[i]) * s_scl[i];
      tr += fabs(g);
      mx = fmax(mx, g);
    }
    for (int o = 32; o > 0; o >>= 1) {
      tr += __shfl_xor(tr, o, 64);
      mx = fmax(mx, __shfl_xor(mx, o, 64));
    }
    if (lane == 0) {
      if (pre) {
        // shift already added; threshold and pivot floor of the whole matrix
        s_zero = 0;
        s_shift = 0.0;
        s_thr = pre[0];
        s_floor = pre[1];
      } else {
        s_zero = !(tr > 0.0);
        s_shift = shift_coef * tr;
        // pivots at or below rel_floor * max diagonal mark a column that is
        // numerically in the span of the previous ones (rank-deficient block)
        s_thr = rel_floor > 0.0 ? rel_floor * (mx + s_shift) : -1.0;
        // floor for pivots that rounding pushed to <= 0 when no deficiency
        // test is requested (first, shifted pass)
        s_floor = s_shift > 0.0 ? s_shift : DBL_MIN;
      }
    }
  }
  __syncthreads();
  if (s_zero) {
    // Zero (or NaN) Gram matrix: the input block is zero.  R = 0 (the block
    // has no range), Rinv = I so that Q = Y * Rinv stays zero.
    for (int r = r0; r < p; r += kCholWaves)
      for (int c = c0; c < p; c += 64) {
        if (R) R[r * p + c] = 0.0;
        Rinv[r * p + c] = (r == c) ? 1.0 : 0.0;
      }
    return;
  }
  // Near-identity Gram matrix (the second pass of a two-pass CholeskyQR):
  // with Gs = I + E, every |E_ij| <= 1e-10 and no shift, the factor is
  // R~ = I + U, U = triu(E) with halved diagonal, and R~^{-1} = I - U, both
  // exact to O(||U||^2) <= 2e-16 (||U||_2 <= 128 * 1e-10): no pivot chain.
  // No pivot can fall to the drop threshold (pivots are 1 +- 1e-10), so the
  // factorisation would drop nothing either.
  if (!pre && shift_coef == 0.0 && s_near) {
#pragma unroll 2
    for (int r = r0; r < p; r += kCholWaves)
#pragma unroll 2
      for (int c = c0; c < p; c += 64) {
        const double e = c > r ? A[r * ld + c] : (c == r ? 0.5 * (A[r * ld + r] - 1.0) : 0.0);
        const double id = r == c ? 1.0 : 0.0;
        if (R) R[r * p + c] = (id + e) * s_dg[c];
        Rinv[r * p + c] = s_scl[r] * (id - e);
      }
    return;
  }
  const double shift = s_shift, thr = s_thr, floor_d = s_floor;
  if (shift != 0.0) {
    for (int i = tid; i < p; i += kCholThreads) A[i * ld + i] += shift;
    __syncthreads();
  }

  // Cholesky of the diagonal block at K0 (one wave): rows of F, reciprocal
  // pivots and dropped-column flags (unit pivot, zero row) to LDS.
  auto factor_diag = [&](int K0) {
    double a[16], rd = 0.0;
    int drop = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = A[(K0 + r) * ld + K0 + lc];
    unroll<16>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      double piv = row_bcast<k>(a[k]);
      const bool dk = thr >= 0.0 && !(piv > thr);
      if (dk || !(piv > floor_d)) piv = floor_d;
      const double rs = rsqrt_newton(piv);
      const double m = dk ? 0.0 : a[k] * rs;
      unroll<16>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        if constexpr (r > k) a[r] = fma(-row_bcast<r>(m), m, a[r]);
      });
      // entries left of the diagonal are meaningless, and never read
      A[(K0 + k) * ld + K0 + lc] = lc == k ? (dk ? 1.0 : piv * rs) : m;
      if (lc == k) {
        rd = dk ? 0.0 : rs;
        drop = dk ? 1 : 0;
      }
    });
    s_rd[K0 + lc] = rd;
    defic[K0 + lc] = drop;
  };
  // A[I0][J0] -= F[K0][I0]^T F[K0][J0]
  auto trail = [&](int K0, int I0, int J0) {
    d4 acc;
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = A[(I0 + lr + 4 * q) * ld + J0 + lc];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const double av = -A[(K0 + 4 * s + lr) * ld + I0 + lc];
      const double bv = A[(K0 + 4 * s + lr) * ld + J0 + lc];
      acc = mfma16(av, bv, acc);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) A[(I0 + lr + 4 * q) * ld + J0 + lc] = acc[q];
  };
  for (int kb = 0; kb < nb; ++kb) {
    int K0 = kb * 16;
    asm volatile("" : "+s"(K0));  // one base address, not one induction variable per row
    const int n = nb - kb - 1;
    // ---- phase B of block column kb - 1 --------------------------------------
    if (w == 0) {
      if (kb > 0) {
        trail(K0 - 16, K0, K0);
        wave_lds_fence();
      }
      factor_diag(K0);
    } else if (kb > 0) {
      for (int t = w; t < (n + 1) * (n + 2) / 2; t += kCholWaves - 1) {
        int bi = 0, rem = t;  // row-wise enumeration of the upper blocks
        while (rem >= n + 1 - bi) {
          rem -= n + 1 - bi;
          ++bi;
        }
        trail(K0 - 16, (kb + bi) * 16, (kb + bi + rem) * 16);
      }
    }
    __syncthreads();
    // ---- phase A -----------------------------------------------------------
    // Block row of F: F_kk^T P = A[K0:K0+16, col], rows of dropped columns
    // set to zero.  Column-oriented: once v_t is final (times 1/F[t][t], 0
    // for a dropped column) it is eliminated from all later rows at once.
    const int ncol = 16 * n;
    if (w * 64 < ncol) {
      double x[16];
      const int col = K0 + 16 + min(tid, ncol - 1);  // idle lanes repeat the last column
      const double rdv = s_rd[K0 + lc];
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] = A[(K0 + r) * ld + col];
      double f = A[K0 * ld + K0 + lc];  // row t of F_kk, one step ahead
      unroll<16>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        const double fn = A[(K0 + (t < 15 ? t + 1 : t)) * ld + K0 + lc];
        x[t] *= row_bcast<t>(rdv);
        unroll<16>([&](auto rc) {
          constexpr int r = decltype(rc)::value;
          if constexpr (r > t) x[r] = fma(-row_bcast<r>(f), x[t], x[r]);
        });
        f = fn;
        // without it all 120 broadcasts are hoisted, and spilled
        __builtin_amdgcn_sched_barrier(0);
      });
      // stores without a guard, here and below: the FMAs would be sunk into
      // the guarded block, away from their broadcasts
#pragma unroll
      for (int r = 0; r < 16; ++r) A[(K0 + r) * ld + col] = x[r];
    } else if (w == kCholWaves - 1) {
      // F_kk^{-1}, lane lc holding column lc, rows from the bottom:
      //   X[i][c] = (delta_ic - sum_{k>i} F[i][k] X[k][c]) / F[i][i].
      // A dropped column i gets a zero row i (and column i) here; no other
      // column of X depends on it (row i of F is e_i^T, so the exact X[i][c]
      // is 0 for c != i).
      double x[16];
      const double rdv = s_rd[K0 + lc];
      int id = lc;
      asm volatile("" : "+v"(id));  // else the unit columns are kept through the loop
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] = id == r ? 1.0 : 0.0;
      double f = A[(K0 + lc) * ld + K0 + 15];  // column i of F_kk, one step ahead
      unroll<16>([&](auto tc) {
        constexpr int i = 15 - decltype(tc)::value;
        const double fn = A[(K0 + lc) * ld + K0 + (i > 0 ? i - 1 : 0)];
        x[i] *= row_bcast<i>(rdv);
        unroll<16>([&](auto rc) {
          constexpr int r = decltype(rc)::value;
          if constexpr (r < i) x[r] = fma(-row_bcast<r>(f), x[i], x[r]);
        });
        f = fn;
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int r = 0; r < 16; ++r) Xd[(K0 + r) * kCholXdLd + lc] = x[r];
    }
    __syncthreads();
  }

  // ---- X = F^{-1}, block column j on one wave, rows from the bottom:
  //   X[bi][j] = -F_bi^{-1} sum_{bi<k<=j} F[bi][k] X[k][j],
  // the sums of all rows in registers, a block's output registers being the
  // B operand of the next products: no barrier, no LDS round trip.  (Back
  // substitution by columns keeps F X - I small, which Y X needs; X computed
  // from X F = I, block column by block column beside the factorisation, lost
  // the orthogonality of Y X to the condition of F.)  The longest and the
  // shortest column share a SIMD.  Blocks of X go transposed below the
  // diagonal.
  {
    const int j = w < 4 ? nb - 1 - w : w - 4;
    if (j > 0 && (w < 4 || j < nb - 4)) {
      d4 T[7], Xc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int bi = 0; bi < 7; ++bi) T[bi] = d4{0.0, 0.0, 0.0, 0.0};
      unroll<7>([&](auto ic) {
        constexpr int k = 7 - decltype(ic)::value;
        if (k <= j) {
          if (k == j) {
#pragma unroll
            for (int s = 0; s < 4; ++s) Xc[s] = Xd[(j * 16 + 4 * s + lr) * kCholXdLd + lc];
          }
          unroll<k>([&](auto bc) {
            constexpr int bi = k - 1 - decltype(bc)::value;
#pragma unroll
            for (int s = 0; s < 4; ++s)
              T[bi] = mfma16(A[(bi * 16 + lc) * ld + k * 16 + 4 * s + lr], Xc[s], T[bi]);
          });
          d4 Xo = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
          for (int s = 0; s < 4; ++s)
            Xo = mfma16(-Xd[((k - 1) * 16 + lc) * kCholXdLd + 4 * s + lr], T[k - 1][s], Xo);
#pragma unroll
          for (int q = 0; q < 4; ++q) A[(j * 16 + lc) * ld + (k - 1) * 16 + lr + 4 * q] = Xo[q];
          Xc = Xo;
        }
      });
    }
  }
  __syncthreads();

#pragma unroll 2
  for (int r = r0; r < p; r += kCholWaves)
#pragma unroll 2
    for (int c = c0; c < p; c += 64) {
      double xv = 0.0;
      // a dropped column gets a zero column in R^{-1}: Q = Y R^{-1} then
      // has an exact zero there instead of an unnormalised residual (the
      // other columns of Q do not depend on it: row c of F is e_c^T)
      if (c >= r && !defic[c])
        xv = (r >> 4) == (c >> 4) ? Xd[r * kCholXdLd + (c & 15)] : A[c * ld + r];
      if (R) R[r * p + c] = (c >= r && !defic[r] ? A[r * ld + c] : 0.0) * s_dg[c];
      Rinv[r * p + c] = xv * s_scl[r];
    }
}

// Cholesky of Gram matrices wider than one LDS-resident factorisation
// (128 < p <= 256), as two 128-blocks: with Gs = D G D + shift I (the
// scaled, shifted matrix of chol_inv_kernel) split at p1,
//   F11 = chol(Gs11), F12 = F11^{-T} Gs12, F22 = chol(Gs22 - F12^T F12),
//   F^{-1} = [X11, -X11 F12 X22; 0, X22]   (X = F^{-1} of each block),
// both block factorisations with the whole matrix's pivot threshold, so
// that a column of the second block that is dependent on the first one is
// dropped as the unblocked factorisation would drop it.
// chol_prep_kernel: scales (D, D^{-1}), shift, threshold and pivot floor,
// and the three blocks of Gs (contiguous, row-major).  A zero (or NaN) Gram
// matrix gives Gs = I with D = 0 and D^{-1} = 1: R = 0, R^{-1} = I.
__global__ __launch_bounds__(1024) void chol_prep_kernel(
    const double *G, int p, int p1, double coef, double rel_floor, double *G11,
    double *G12, double *G22, double *dg, double *scl, double *params) {
  __shared__ double s_scl[256];
  __shared__ double s_tr[16], s_mx[16];
  __shared__ double s_shift;
  __shared__ int s_zero;
  const int tid = threadIdx.x;
  const int p2 = p - p1;
  double tr = 0.0, mx = 0.0;
  for (int i = tid; i < p; i += blockDim.x) {
    const double g = G[(int64_t)i * p + i];
    const double d = g > 0.0 ? sqrt(g) : 0.0;
    const double sc = d > 0.0 ? 1.0 / d : 0.0;
    s_scl[i] = sc;
    const double gs = (g * sc) * sc;
    tr += fabs(gs);
    mx = fmax(mx, gs);
  }
  for (int o = 32; o > 0; o >>= 1) {
    tr += __shfl_xor(tr, o, 64);
    mx = fmax(mx, __shfl_xor(mx, o, 64));
  }
  if ((tid & 63) == 0) {
    s_tr[tid >> 6] = tr;
    s_mx[tid >> 6] = mx;
  }
  __syncthreads();
  if (tid == 0) {
    double t = 0.0, x = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
      t += s_tr[w];
      x = fmax(x, s_mx[w]);
    }
    const int zero = !(t > 0.0);
    const double shift = coef * t;
    s_zero = zero;
    s_shift = zero ? 0.0 : shift;
    params[0] = rel_floor > 0.0 ? rel_floor * (x + shift) : -1.0;
    params[1] = shift > 0.0 ? shift : DBL_MIN;
  }
  __syncthreads();
  const int zero = s_zero;
  const double shift = s_shift;
  for (int i = tid; i < p; i += blockDim.x) {
    const double sc = s_scl[i];
    dg[i] = zero ? 0.0 : (sc > 0.0 ? 1.0 / sc : 0.0);
    scl[i] = zero ? 1.0 : sc;
  }
  for (int e = tid; e < p * p; e += blockDim.x) {
    const int r = e / p, c = e - (e / p) * p;
    const double v = zero ? (r == c ? 1.0 : 0.0)
                          : (G[e] * s_scl[r]) * s_scl[c] + (r == c ? shift : 0.0);
    if (r < p1) {
      if (c < p1)
        G11[r * p1 + c] = v;
      else
        G12[r * p2 + c - p1] = v;
    } else if (c >= p1) {
      G22[(r - p1) * p2 + c - p1] = v;
    }
  }
}

// F12 = F11^{-T} G12 by forward substitution (backward stable, unlike the
// product with the explicit inverse X11^T, whose error grows with cond(F11)
// and is large exactly where the block's columns are nearly dependent).  F11
// is the upper factor as chol_inv_upper writes it (a dropped column has a
// zero row, diagonal included; its row of F12 is zero).  One workgroup,
// F11 in LDS, one thread per column of G12 holding that column in
// registers, right-looking: v_t /= F[t][t], then v_r -= F[t][r] v_t for all
// r > t (independent updates, the F entries LDS broadcasts).
constexpr int kTrsmRows = 128;

__global__ __launch_bounds__(128) void trsm_ut_kernel(const double *F, int p2,
                                                      const double *G, double *V) {
  constexpr int n = kTrsmRows;
  extern __shared__ double Fs[];  // n x (n + 1)
  const int tid = threadIdx.x;
  for (int e = tid; e < n * n; e += blockDim.x) {
    const int r = e / n, c = e - (e / n) * n;
    Fs[r * (n + 1) + c] = F[e];
  }
  __syncthreads();
  if (tid >= p2) return;
  double v[n];
#pragma unroll
  for (int r = 0; r < n; ++r) v[r] = G[(int64_t)r * p2 + tid];
#pragma unroll
  for (int t = 0; t < n; ++t) {
    const double d = Fs[t * (n + 1) + t];
    v[t] = d != 0.0 ? v[t] / d : 0.0;
#pragma unroll
    for (int r = t + 1; r < n; ++r) v[r] -= Fs[t * (n + 1) + r] * v[t];
  }
#pragma unroll
  for (int r = 0; r < n; ++r) V[(int64_t)r * p2 + tid] = v[r];
}

// R and R^{-1} in the unscaled basis: R[r][c] = F[r][c] dg[c],
// R^{-1}[r][c] = scl[r] X[r][c], from the blocks (U = X11 F12 X22).
__global__ void chol_assemble_kernel(int p, int p1, const double *F11,
                                     const double *X11, const double *F12,
                                     const double *U, const double *F22,
                                     const double *X22, const double *dg,
                                     const double *scl, double *R, double *Rinv) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= p * p) return;
  const int r = e / p, c = e - (e / p) * p;
  const int p2 = p - p1;
  double f = 0.0, x = 0.0;
  if (r < p1) {
    if (c < p1) {
      f = F11[r * p1 + c];
      x = X11[r * p1 + c];
    } else {
      f = F12[r * p2 + c - p1];
      x = -U[r * p2 + c - p1];
    }
  } else if (c >= p1) {
    f = F22[(r - p1) * p2 + c - p1];
    x = X22[(r - p1) * p2 + c - p1];
  }
  if (R) R[e] = f * dg[c];
  Rinv[e] = scl[r] * x;
}

// ---------------------------------------------------------------------------
// One-sided Jacobi SVD.
// ---------------------------------------------------------------------------
// Cross-lane moves inside a 16-lane row with DPP (register-to-register, no
// LDS round trip): quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror,
// row_mirror.  Each pairs every lane with one of the other half of the group
// being combined, so four steps give every lane the sum over its 16 lanes.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double sum16(double v) {
  v += dpp_f64<0xB1>(v);
  v += dpp_f64<0x4E>(v);
  v += dpp_f64<0x141>(v);
  v += dpp_f64<0x140>(v);
  return v;
}

// Pivoted Householder QR of A^T (A: m x n row-major, m, n <= 128, one
// workgroup) as the preconditioner of the one-sided Jacobi SVD:
//   A = W Q^T, Q (n x r) orthonormal, W = A Q (m x r), r = min(m, n).
// W is lower triangular up to the order of its rows, with columns of falling
// length, and its columns are close to orthogonal: the Jacobi needs 5 to 7
// sweeps on it where the projector matrices of a D=2, chi=10 run (40 x 40,
// graded over 11 decades) took 15 to 17, and r columns instead of n.  A row of A is a
// column of A^T, so the pivot is the longest remaining row, and no row is
// moved: used rows keep their Householder vector.  64 groups of 16 lanes, a
// row per group; one barrier per step (the norms of the rows' remainders,
// recomputed in the update, pick the next pivot in every wave).  On those 40 x 40
// matrices it costs 90 us, and Jacobi and replay fall from 720 + 219 to
// 228 + 18 us.
constexpr int kQrpThreads = 1024;
// smallest squared norm of a remainder that is still reflected (the matrix
// scaled to a largest entry in [1, 2))
constexpr double kQrpNull = 1e-280;

__global__ __launch_bounds__(kQrpThreads) void qrp_kernel(const double *A, int m, int n,
                                                          double *W, double *Q) {
  extern __shared__ double S[];  // m rows of n, padded to ld
  __shared__ double s_nrm[2][kMaxDim];  // squared norm of the rest, -1: used
  __shared__ double s_tau[kMaxDim], s_head[kMaxDim], s_alpha[kMaxDim];
  __shared__ double s_big[kQrpThreads / 64];
  __shared__ int s_piv[kMaxDim], s_pos[kMaxDim];
  constexpr int NG = kQrpThreads / 16;
  const int ld = n | 1;
  const int r = min(m, n);
  const int tid = threadIdx.x, lane = tid & 63;
  const int grp = tid >> 4, gl = tid & 15;
  bool finite = true;
  double big = 0.0;
  for (int e = tid; e < m * n; e += kQrpThreads) {
    const int j = e / n;
    const double v = A[e];
    finite = finite && fabs(v) <= DBL_MAX;
    big = fmax(big, fabs(v));
    S[j * ld + (e - j * n)] = v;
  }
  for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
  if (lane == 0) s_big[tid >> 6] = big;
  if (tid < m) s_pos[tid] = r;
  // a NaN or infinite entry: every value and vector of this matrix is NaN
  // (below, a NaN norm would be taken for the norm of a zero row)
  if (__syncthreads_or(!finite)) {
    const double nan = __builtin_nan("");
    for (int e = tid; e < m * r; e += kQrpThreads) W[e] = nan;
    for (int e = tid; e < n * r; e += kQrpThreads) Q[e] = nan;
    return;
  }
  // scaled by a power of two (exact) to a largest entry in [1, 2), as in
  // jacobi_kernel: the squared norms do not overflow, and vanish only for rows
  // 1e-154 times the largest entry
  for (int w = 0; w < kQrpThreads / 64; ++w) big = fmax(big, s_big[w]);
  const int ex = big > 0.0 ? __builtin_amdgcn_frexp_exp(big) - 1 : 0;
  for (int e = tid; e < m * n; e += kQrpThreads) {  // the elements this thread stored
    const int j = e / n;
    double &x = S[j * ld + (e - j * n)];
    x = __builtin_amdgcn_ldexp(x, -ex);
  }
  __syncthreads();
  for (int j = grp; j < m; j += NG) {
    double acc = 0.0;
    for (int i = gl; i < n; i += 16) acc = fma(S[j * ld + i], S[j * ld + i], acc);
    acc = sum16(acc);
    if (gl == 0) s_nrm[0][j] = acc;
  }
  __syncthreads();
  int done = 0;  // reflections made
  for (int k = 0; k < r; ++k) {
    const double *cur = s_nrm[k & 1];
    double *next = s_nrm[(k + 1) & 1];
    // the longest remaining row (the smallest index on a tie)
    double best = lane < m ? cur[lane] : -2.0;
    int bj = lane;
    if (lane + 64 < m && cur[lane + 64] > best) {
      best = cur[lane + 64];
      bj = lane + 64;
    }
    for (int o = 32; o > 0; o >>= 1) {
      const double ov = __shfl_xor(best, o, 64);
      const int oj = __shfl_xor(bj, o, 64);
      if (ov > best || (ov == best && oj < bj)) {
        best = ov;
        bj = oj;
      }
    }
    bj = __builtin_amdgcn_readfirstlane(bj);
    // What remains is zero, or too small for 1 / (squared norm): no more
    // reflections.  The rows not used keep their entries (past column r they
    // are dropped, 1e-140 of the largest).
    if (!(best > kQrpNull)) break;
    done = k + 1;
    // Householder vector of its elements k..n-1 (in place; the head apart)
    const double *v = S + bj * ld;
    const double bk = v[k];
    const double nb = sqrt(best);
    const double al = bk > 0.0 ? -nb : nb;
    const double head = bk - al;
    const double tau = 1.0 / (best + fabs(bk) * nb);
    if (tid == 0) {
      s_tau[k] = tau;
      s_head[k] = head;
      s_alpha[k] = al;
      s_piv[k] = bj;
      s_pos[bj] = k;
    }
    const int i0 = (k & ~15) + gl;
    for (int j = grp; j < m; j += NG) {
      const bool live = j != bj && cur[j] >= 0.0;
      if (live) {
        double *b = S + j * ld;
        double dot = 0.0;
        for (int i = i0; i < n; i += 16) {
          const double vi = i == k ? head : v[i];
          if (i >= k) dot = fma(vi, b[i], dot);
        }
        const double f = tau * sum16(dot);
        double rest = 0.0;
        for (int i = i0; i < n; i += 16) {
          const double vi = i == k ? head : v[i];
          if (i >= k) {
            const double x = fma(-f, vi, b[i]);
            b[i] = x;
            if (i > k) rest = fma(x, x, rest);
          }
        }
        rest = sum16(rest);
        if (gl == 0) next[j] = rest;
      } else if (gl == 0) {
        next[j] = -1.0;
      }
    }
    __syncthreads();
  }
  // W, column-major: row j holds R's entries up to its pivot step
  for (int e = tid; e < m * r; e += kQrpThreads) {
    const int c = e / m, j = e - c * m;
    const int pos = s_pos[j];
    W[e] = c < pos ? __builtin_amdgcn_ldexp(S[j * ld + c], ex)
                   : (c == pos ? __builtin_amdgcn_ldexp(s_alpha[c], ex) : 0.0);
  }
  // Q = H_0 ... H_{r-1} (unit columns): column c on one group, in registers
  for (int c = grp; c < r; c += NG) {
    double q[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) q[u] = gl + 16 * u == c ? 1.0 : 0.0;
    for (int k = min(c, done - 1); k >= 0; --k) {
      const double *v = S + s_piv[k] * ld;
      const double head = s_head[k];
      double vv[8], dot = 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i = gl + 16 * u;
        vv[u] = i < k || i >= n ? 0.0 : (i == k ? head : v[i]);
        dot = fma(vv[u], q[u], dot);
      }
      const double f = s_tau[k] * sum16(dot);
#pragma unroll
      for (int u = 0; u < 8; ++u) q[u] = fma(-f, vv[u], q[u]);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (gl + 16 * u < n) Q[(int64_t)(gl + 16 * u) * r + c] = q[u];
  }
}

// Round-robin (circle method) pairing for pe (even) players, round s:
// pair 0 = (s, pe-1); pair k>0 = ((s+k) mod (pe-1), (s-k) mod (pe-1)).
__device__ __forceinline__ void rr_pair(int s, int k, int pe, int &i, int &j) {
  // 0 <= s, k < q: the residues mod q need one conditional subtraction each
  // (no integer division in the rotation loops)
  const int q = pe - 1;
  if (k == 0) {
    i = s;
    j = q;
  } else {
    i = s + k;
    if (i >= q) i -= q;
    j = s - k;
    if (j < 0) j += q;
  }
  if (i > j) {
    const int t = i;
    i = j;
    j = t;
  }
}

// The rotation that makes columns of squared norms a, bb and inner product g
// orthogonal (x' = c x - s y, y' = s x + c y): with d = bb - a,
//   cos 2t = |d| / sqrt(d^2 + 4 g^2), c^2 = (1 + cos 2t) / 2,
//   s = sign(d) g / (c sqrt(d^2 + 4 g^2)).
// Two reciprocal square roots instead of two square roots and two divisions
// (the angle is computed by all 16 lanes of a pair, so it weighs as much as
// the rotation itself); scaled to a + bb ~ 1 so that the squares neither
// overflow nor vanish.
__device__ __forceinline__ void jacobi_angle(double a, double bb, double g, double &c,
                                             double &s) {
  const int e = -__builtin_amdgcn_frexp_exp(a + bb);
  const double d = __builtin_amdgcn_ldexp(bb - a, e), gs = __builtin_amdgcn_ldexp(g, e);
  const double r1 = rsqrt_newton(fma(d, d, 4.0 * gs * gs));
  const double c2 = fma(0.5 * fabs(d), r1, 0.5);
  const double r2 = rsqrt_newton(c2);
  c = c2 * r2;
  s = (d < 0.0 ? -gs : gs) * r1 * r2;
}

// FULL: m == kMaxDim (the randomized path's projected problems), so the
// row guards of the inner loops are compile-time true.
template <bool FULL>
__global__ __launch_bounds__(1024) void jacobi_kernel(
    double *Wg, int m_arg, int p, double tol, int max_sweeps, double *sigma,
    double *rot, int *nsteps) {
  const int m = FULL ? kMaxDim : m_arg;
  extern __shared__ double W[];  // pe columns of length m (col-major)
  __shared__ double s_off[64];
  __shared__ double s_tiny;
  const int b = blockIdx.x;
  double *Wb = Wg + (int64_t)b * m * p;
  const int pe = p + (p & 1);  // even number of columns (pad one zero col)
  const int tid = threadIdx.x;
  const int nt = blockDim.x;
  double big = 0.0;
  for (int i0 = 0; i0 < m * pe; i0 += 8 * nt) {  // 8 loads in flight
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + u * nt + tid;
      v[u] = (i < m * p) ? Wb[i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + u * nt + tid;
      if (i < m * pe) W[i] = v[u];
      big = fmax(big, fabs(v[u]));
    }
  }
  // scaled by a power of two (exact) to a largest entry in [1, 2): the
  // products of squared norms in the convergence test neither overflow nor
  // vanish
  for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
  if ((tid & 63) == 0) s_off[tid >> 6] = big;
  __syncthreads();
  for (int w = 0; w < (nt >> 6); ++w) big = fmax(big, s_off[w]);
  const int ex = big > 0.0 && big <= DBL_MAX ? __builtin_amdgcn_frexp_exp(big) - 1 : 0;
  __syncthreads();
  double fro = 0.0;
  for (int i = tid; i < m * pe; i += nt) {  // the elements this thread stored
    const double v = __builtin_amdgcn_ldexp(W[i], -ex);
    W[i] = v;
    fro += v * v;
  }
  for (int o = 32; o > 0; o >>= 1) fro += __shfl_xor(fro, o, 64);
  if ((tid & 63) == 0) s_off[tid >> 6] = fro;
  __syncthreads();
  if (tid == 0) {
    double f = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) f += s_off[w];
    // columns whose norm is below 1e-30 of the matrix norm are treated as
    // zero: neither rotated nor counted for convergence.  The bound is far
    // below rounding level on purpose: skipping a column of norm t leaves a
    // kept column of norm s unrotated by an angle of up to t / s, and kept
    // singular values go down to 1e-12 of the largest.
    s_tiny = f * 1e-60;
  }
  __syncthreads();
  const double tiny = s_tiny;
  const double tol2 = tol * tol;

  const int grp = tid >> 4;  // pair slot 0..63
  const int gl = tid & 15;   // lane in the 16-lane group
  const int npairs = pe / 2;
  const int64_t rot_stride = (int64_t)max_sweeps * (pe - 1) * npairs * 2;
  double *rotb = rot ? rot + (int64_t)b * rot_stride : nullptr;
  int steps = 0;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    double off_local = 0.0;
    for (int s = 0; s < pe - 1; ++s) {
      for (int k = grp; k < npairs; k += 64) {
        int i, j;
        rr_pair(s, k, pe, i, j);
        double *wi = W + i * m;
        double *wj = W + j * m;
        // the pair's two columns stay in registers between the inner
        // products and the rotation (m <= 128: 8 rows per lane)
        double xr[8], yr[8];
        double a = 0.0, bb = 0.0, g = 0.0;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int r = gl + 16 * u;
          xr[u] = (FULL || r < m) ? wi[r] : 0.0;
          yr[u] = (FULL || r < m) ? wj[r] : 0.0;
          a += xr[u] * xr[u];
          bb += yr[u] * yr[u];
          g += xr[u] * yr[u];
        }
        a = sum16(a);
        bb = sum16(bb);
        g = sum16(g);
        double c = 1.0, sn = 0.0;
        // rotate when |g| / sqrt(a bb) > tol, tested without a division
        const double g2 = g * g;
        if (g != 0.0 && a > tiny && bb > tiny && g2 > tol2 * (a * bb)) {
          {
            off_local = 1.0;
            jacobi_angle(a, bb, g, c, sn);
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              const int r = gl + 16 * u;
              if (FULL || r < m) {
                wi[r] = c * xr[u] - sn * yr[u];
                wj[r] = sn * xr[u] + c * yr[u];
              }
            }
          }
        }
        if (rotb && gl == 0) {
          double *dst = rotb + ((int64_t)steps * npairs + k) * 2;
          dst[0] = c;
          dst[1] = sn;
        }
      }
      ++steps;
      __syncthreads();
    }
    // did any pair of this sweep exceed the tolerance (off_local = 1)?
    double v = off_local;
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    if ((tid & 63) == 0) s_off[tid >> 6] = v;
    __syncthreads();
    double off = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) off = fmax(off, s_off[w]);
    __syncthreads();
    if (!(off > 0.0)) break;
  }
  for (int jc = tid; jc < p; jc += blockDim.x) {
    double acc = 0.0;
    const double *wc = W + jc * m;
    for (int r = 0; r < m; ++r) acc += wc[r] * wc[r];
    sigma[(int64_t)b * p + jc] = __builtin_amdgcn_ldexp(sqrt(acc), ex);
  }
  for (int i = tid; i < m * p; i += blockDim.x) Wb[i] = __builtin_amdgcn_ldexp(W[i], ex);
  if (tid == 0 && nsteps) nsteps[b] = steps;
}

// One-sided Jacobi for matrices of up to kMaxDimBig columns and rows that
// do not fit in LDS: the same round-robin rounds, rotation formula,
// convergence test and rotation stream as jacobi_kernel, with the matrix
// in global memory (it stays in L2: 512 KB at 256 x 256).  One workgroup per
// matrix, 64 groups of 16 lanes, each group one column pair per step (the
// two columns in registers, 16 rows per lane); the workgroup barrier
// between rounds orders the rounds' global reads after the previous round's
// writes (all waves of a workgroup share one CU's cache).
constexpr int kMaxDimBig = 256;

__global__ __launch_bounds__(1024) void jacobi_big_kernel(
    double *Wg, int m, int p, double tol, int max_sweeps, double *sigma,
    double *rot, int *nsteps) {
  __shared__ double s_off[16];
  __shared__ double s_tiny;
  const int b = blockIdx.x;
  double *W = Wg + (int64_t)b * m * p;
  const int pe = p + (p & 1);
  const int tid = threadIdx.x;
  // A largest entry outside [2^-100, 2^100] is scaled by a power of two
  // (exact), as in jacobi_kernel; between them the squared norms down to the
  // 1e-60 of s_tiny and their products with tol^2 stay in range, and the
  // pass over global memory is saved.
  double fro = 0.0, big = 0.0;
  for (int i = tid; i < m * p; i += blockDim.x) {
    fro += W[i] * W[i];
    big = fmax(big, fabs(W[i]));
  }
  for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
  if ((tid & 63) == 0) s_off[tid >> 6] = big;
  __syncthreads();
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) big = fmax(big, s_off[w]);
  __syncthreads();
  int ex = big > 0.0 && big <= DBL_MAX ? __builtin_amdgcn_frexp_exp(big) - 1 : 0;
  if (ex >= -100 && ex <= 100) ex = 0;
  if (ex != 0) {
    fro = 0.0;
    for (int i = tid; i < m * p; i += blockDim.x) {
      const double v = __builtin_amdgcn_ldexp(W[i], -ex);
      W[i] = v;
      fro += v * v;
    }
  }
  for (int o = 32; o > 0; o >>= 1) fro += __shfl_xor(fro, o, 64);
  if ((tid & 63) == 0) s_off[tid >> 6] = fro;
  __syncthreads();
  if (tid == 0) {
    double f = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) f += s_off[w];
    s_tiny = f * 1e-60;  // as in jacobi_kernel
  }
  __syncthreads();
  const double tiny = s_tiny;
  const double tol2 = tol * tol;
  const int grp = tid >> 4;
  const int gl = tid & 15;
  const int npairs = pe / 2;
  const int64_t rot_stride = (int64_t)max_sweeps * (pe - 1) * npairs * 2;
  double *rotb = rot ? rot + (int64_t)b * rot_stride : nullptr;
  int steps = 0;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    double off_local = 0.0;
    for (int s = 0; s < pe - 1; ++s) {
      for (int k = grp; k < npairs; k += 64) {
        int i, j;
        rr_pair(s, k, pe, i, j);
        // the padding column (p odd) is zero: its pairs never rotate
        const bool real_j = j < p;
        double *wi = W + (int64_t)i * m;
        double *wj = W + (int64_t)j * m;
        double xr[16], yr[16];
        double a = 0.0, bb = 0.0, g = 0.0;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int r = gl + 16 * u;
          xr[u] = r < m ? wi[r] : 0.0;
          yr[u] = (real_j && r < m) ? wj[r] : 0.0;
          a += xr[u] * xr[u];
          bb += yr[u] * yr[u];
          g += xr[u] * yr[u];
        }
        a = sum16(a);
        bb = sum16(bb);
        g = sum16(g);
        double c = 1.0, sn = 0.0;
        const double g2 = g * g;
        if (g != 0.0 && a > tiny && bb > tiny && g2 > tol2 * (a * bb)) {
          off_local = 1.0;
          jacobi_angle(a, bb, g, c, sn);
#pragma unroll
          for (int u = 0; u < 16; ++u) {
            const int r = gl + 16 * u;
            if (r < m) {
              wi[r] = c * xr[u] - sn * yr[u];
              wj[r] = sn * xr[u] + c * yr[u];
            }
          }
        }
        if (rotb && gl == 0) {
          double *dst = rotb + ((int64_t)steps * npairs + k) * 2;
          dst[0] = c;
          dst[1] = sn;
        }
      }
      ++steps;
      __syncthreads();
    }
    double v = off_local;
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    if ((tid & 63) == 0) s_off[tid >> 6] = v;
    __syncthreads();
    double off = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) off = fmax(off, s_off[w]);
    __syncthreads();
    if (!(off > 0.0)) break;
  }
  for (int jc = tid; jc < p; jc += blockDim.x) {
    double acc = 0.0;
    const double *wc = W + (int64_t)jc * m;
    for (int r = 0; r < m; ++r) acc += wc[r] * wc[r];
    sigma[(int64_t)b * p + jc] = __builtin_amdgcn_ldexp(sqrt(acc), ex);
  }
  if (ex != 0) {
    __syncthreads();  // the norms above read the columns
    for (int i = tid; i < m * p; i += blockDim.x) W[i] = __builtin_amdgcn_ldexp(W[i], ex);
  }
  if (tid == 0 && nsteps) nsteps[b] = steps;
}

// J = J0 * (product of recorded rotations), p <= 128 columns, J0 (rows x p)
// given or the identity.  The rows of J are independent: one wave carries a
// row, lane k the two elements of the round's pair k.  From one round-robin round to the next the first elements of the
// pairs move one lane down and the second ones one lane up (the last lane
// turns its second into a first, lane 0 its first into lane 1's second and
// keeps the fixed column), so a round is four FMAs, one coalesced load of its
// (c, s) a chunk of rounds ahead, and DPP wave shifts: no LDS and no barrier.
// 128 rows, 762 rounds: 43 us against 209 us with the rows in LDS.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

__global__ __launch_bounds__(64) void jacobi_replay_kernel(const double *rot, const int *nsteps,
                                                           int p, const double *J0, double *J) {
  constexpr int CH = 8;  // rounds per chunk of loads
  constexpr int kShl = 0x130, kShr = 0x138;  // lane k from k + 1, from k - 1
  const int np = (p + 1) / 2, q = 2 * np - 1;  // pairs; players but the fixed one
  const int lane = threadIdx.x, row = blockIdx.x;
  const bool first = lane == 0, last = lane == np - 1;
  // round 0: pair k = (k, q - k), pair 0 = (0, q)
  int ia = lane, ib = lane == 0 ? q : q - lane;
  double xa, xb;
  if (J0) {
    const double *j0 = J0 + (int64_t)row * p;
    xa = lane < np && ia < p ? j0[ia] : 0.0;
    xb = lane < np && ib < p ? j0[ib] : 0.0;
  } else {
    xa = ia == row ? 1.0 : 0.0;
    xb = ib == row ? 1.0 : 0.0;
  }
  const int ns = __builtin_amdgcn_readfirstlane(nsteps[0]);
  const double2 *cs = reinterpret_cast<const double2 *>(rot) + min(lane, np - 1);
  double2 nxt[CH];
  auto fetch = [&](int s0) {
#pragma unroll
    for (int u = 0; u < CH; ++u) nxt[u] = cs[(int64_t)min(s0 + u, ns - 1) * np];
  };
  auto round = [&](const double2 &r) {
    // the stream's rotations act on (smaller, larger) column index
    const double sn = ia < ib ? r.y : -r.y;
    const double a = xa;
    xa = fma(r.x, a, -(sn * xb));
    xb = fma(sn, a, r.x * xb);
    const double up = dpp_move<kShr>(first ? xa : xb), down = dpp_move<kShl>(xa);
    xa = np == 1 ? xa : last ? xb : down;
    xb = first ? xb : up;
    const int iup = __builtin_amdgcn_mov_dpp(first ? ia : ib, kShr, 0xF, 0xF, true);
    const int idown = __builtin_amdgcn_mov_dpp(ia, kShl, 0xF, 0xF, true);
    ia = np == 1 ? ia : last ? ib : idown;
    ib = first ? ib : iup;
  };
  if (ns > 0) fetch(0);
  int s0 = 0;
  for (; s0 + CH <= ns; s0 += CH) {
    double2 cur[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) cur[u] = nxt[u];
    fetch(s0 + CH);
#pragma unroll
    for (int u = 0; u < CH; ++u) round(cur[u]);
  }
#pragma unroll
  for (int u = 0; u < CH; ++u)
    if (s0 + u < ns) round(nxt[u]);
  if (lane < np) {
    if (ia < p) J[(int64_t)row * p + ia] = xa;
    if (ib < p) J[(int64_t)row * p + ib] = xb;
  }
}

// The same for 128 < p <= 256.  Row-parallel: one 64-lane
// workgroup owns ROWS rows of J in LDS and replays the rotation stream.  The
// stream is read in chunks of kAccChunk rounds: the next chunk is loaded
// into registers (independent loads, all in flight) while the current one is
// replayed from LDS, so the replay does not wait on memory every round.
constexpr int kAccChunk = 16;

template <int ROWS, int MAXD>
__global__ __launch_bounds__(64) void jacobi_accum_kernel(const double *rot,
                                                          const int *nsteps,
                                                          int p, double *J) {
  __shared__ double row[ROWS][MAXD + 2];
  __shared__ double cs[kAccChunk * (MAXD / 2) * 2];
  const int pe = p + (p & 1);
  const int npairs = pe / 2;
  const int r0 = blockIdx.x * ROWS;
  const int lane = threadIdx.x;
  for (int q = 0; q < ROWS; ++q)
    for (int c = lane; c < pe; c += 64)
      row[q][c] = (r0 + q < p && c == r0 + q) ? 1.0 : 0.0;
  const int ns = nsteps[0];
  const int per = kAccChunk * npairs * 2;  // doubles per chunk (<= 4096)
  const int64_t total = (int64_t)ns * npairs * 2;
  const int nchunks = (ns + kAccChunk - 1) / kAccChunk;
  constexpr int kPerLane = kAccChunk * (MAXD / 2) * 2 / 64;
  double buf[kPerLane];
  auto fetch = [&](int ch) {
    const int64_t base = (int64_t)ch * per;
#pragma unroll
    for (int u = 0; u < kPerLane; ++u) {
      const int idx = u * 64 + lane;
      buf[u] = (idx < per && base + idx < total) ? rot[base + idx] : 0.0;
    }
  };
  if (nchunks > 0) fetch(0);
  int s = 0;  // round-robin step of round st: st mod (pe - 1)
  for (int ch = 0; ch < nchunks; ++ch) {
    __syncthreads();  // the previous chunk has been replayed
#pragma unroll
    for (int u = 0; u < kPerLane; ++u) {
      const int idx = u * 64 + lane;
      if (idx < per) cs[idx] = buf[u];
    }
    __syncthreads();
    if (ch + 1 < nchunks) fetch(ch + 1);
    const int st0 = ch * kAccChunk;
    const int st1 = min(ns, st0 + kAccChunk);
    for (int st = st0; st < st1; ++st, s = (s + 1 == pe - 1) ? 0 : s + 1) {
      const double *cst = cs + (st - st0) * npairs * 2;
      for (int k = lane; k < npairs; k += 64) {
        int i, j;
        rr_pair(s, k, pe, i, j);
        const double c = cst[2 * k];
        const double sn = cst[2 * k + 1];
        // all rows' reads in flight before the first write (the rows are
        // distinct, so the writes cannot feed these reads)
        double x[ROWS], y[ROWS];
#pragma unroll
        for (int q = 0; q < ROWS; ++q) {
          x[q] = row[q][i];
          y[q] = row[q][j];
        }
#pragma unroll
        for (int q = 0; q < ROWS; ++q) {
          row[q][i] = c * x[q] - sn * y[q];
          row[q][j] = sn * x[q] + c * y[q];
        }
      }
      __syncthreads();
    }
  }
  __syncthreads();
  for (int q = 0; q < ROWS; ++q)
    if (r0 + q < p)
      for (int c = lane; c < p; c += 64) J[(int64_t)(r0 + q) * p + c] = row[q][c];
}

// Ranks by counting, one workgroup per list.  The keys are read once into LDS:
// a thread's chain of p loads is what bounds it (p = 128: 12 us from global
// memory, 5 us from LDS).
__global__ __launch_bounds__(128) void sort_desc_kernel(const double *sigma, int p, int batch,
                                                        double *sorted, int *perm) {
  __shared__ double key[kMaxDimBig];
  const int b = blockIdx.x;
  const double *sv = sigma + (int64_t)b * p;
  for (int j = threadIdx.x; j < p; j += blockDim.x) key[j] = rank_key(sv[j]);
  __syncthreads();
  for (int j = threadIdx.x; j < p; j += blockDim.x) {
    const double v = key[j];
    int rank = 0;
    for (int k = 0; k < p; ++k) rank += ranks_before(key[k], k, v, j);
    sorted[(int64_t)b * p + rank] = sv[j];
    perm[(int64_t)b * p + rank] = j;
  }
}

}  // namespace

int jacobi_max_dim() { return kMaxDimBig; }
int jacobi_lds_dim() { return kMaxDim; }

void linalg_init_device() {
  const int lds = kMaxDim * kMaxDim * (int)sizeof(double);
  TN_HIP_CHECK(hipFuncSetAttribute(
      reinterpret_cast<const void *>(&chol_inv_kernel<true>),
      hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)chol_lds_bytes(kMaxDim)));
  TN_HIP_CHECK(hipFuncSetAttribute(
      reinterpret_cast<const void *>(&chol_inv_kernel<false>),
      hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)chol_lds_bytes(kMaxDim)));
  TN_HIP_CHECK(hipFuncSetAttribute(
      reinterpret_cast<const void *>(&jacobi_kernel<true>),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  TN_HIP_CHECK(hipFuncSetAttribute(
      reinterpret_cast<const void *>(&jacobi_kernel<false>),
      hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  TN_HIP_CHECK(hipFuncSetAttribute(
      reinterpret_cast<const void *>(&qrp_kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)((size_t)kMaxDim * (kMaxDim + 1) * sizeof(double))));
  TN_HIP_CHECK(hipFuncSetAttribute(
      reinterpret_cast<const void *>(&trsm_ut_kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)((size_t)kTrsmRows * (kTrsmRows + 1) * sizeof(double))));
}

void randn(double *p, int64_t n, uint64_t seed, uint64_t counter,
           hipStream_t s) {
  if (n <= 0) return;
  int64_t g = (n + 255) / 256;
  if (g > 4096) g = 4096;
  hipLaunchKernelGGL(randn_kernel, dim3((int)g), dim3(256), 0, s, p, n, seed,
                     counter);
  TN_HIP_CHECK(hipGetLastError());
}

void refill_columns(double *X, int64_t n, int p, const double *sigma,
                    double rel, uint64_t seed, uint64_t counter,
                    hipStream_t s) {
  if (n <= 0 || p <= 0) return;
  hipLaunchKernelGGL(refill_columns_kernel, dim3(p), dim3(256), 0, s, X, n, p,
                     sigma, rel, seed, counter);
  TN_HIP_CHECK(hipGetLastError());
}

void chol_inv_upper(const double *G, int p, double shift_coef,
                    double rel_floor, double *R, double *Rinv, hipStream_t s,
                    const double *pre) {
  TN_REQUIRE(p >= 1 && p <= kMaxDim, "chol_inv_upper: p out of range");
  const size_t lds = chol_lds_bytes(p);
  if (p == kMaxDim)
    hipLaunchKernelGGL((chol_inv_kernel<true>), dim3(1), dim3(kCholThreads), lds, s, G, p,
                       shift_coef, rel_floor, R, Rinv, pre);
  else
    hipLaunchKernelGGL((chol_inv_kernel<false>), dim3(1), dim3(kCholThreads), lds, s, G, p,
                       shift_coef, rel_floor, R, Rinv, pre);
  TN_HIP_CHECK(hipGetLastError());
}

int chol_block_dim() { return kMaxDim; }

void trsm_upper_t(const double *F, int p2, const double *G, double *V, hipStream_t s) {
  TN_REQUIRE(p2 >= 1 && p2 <= kTrsmRows, "trsm_upper_t: p2 out of range");
  const size_t lds = (size_t)kTrsmRows * (kTrsmRows + 1) * sizeof(double);
  hipLaunchKernelGGL(trsm_ut_kernel, dim3(1), dim3(128), lds, s, F, p2, G, V);
  TN_HIP_CHECK(hipGetLastError());
}

void chol_prep(const double *G, int p, int p1, double coef, double rel_floor,
               double *G11, double *G12, double *G22, double *dg, double *scl,
               double *params, hipStream_t s) {
  TN_REQUIRE(p > p1 && p1 >= 1 && p <= 256, "chol_prep: sizes out of range");
  hipLaunchKernelGGL(chol_prep_kernel, dim3(1), dim3(1024), 0, s, G, p, p1, coef,
                     rel_floor, G11, G12, G22, dg, scl, params);
  TN_HIP_CHECK(hipGetLastError());
}

void chol_assemble(int p, int p1, const double *F11, const double *X11,
                   const double *F12, const double *U, const double *F22,
                   const double *X22, const double *dg, const double *scl,
                   double *R, double *Rinv, hipStream_t s) {
  TN_REQUIRE(p > p1 && p1 >= 1 && p <= 256, "chol_assemble: sizes out of range");
  hipLaunchKernelGGL(chol_assemble_kernel, dim3(ceil_div(p * p, 256)), dim3(256), 0, s,
                     p, p1, F11, X11, F12, U, F22, X22, dg, scl, R, Rinv);
  TN_HIP_CHECK(hipGetLastError());
}

void jacobi_svd(double *W, int m, int p, int batch, double tol,
                int max_sweeps, double *sigma, double *rot, int *nsteps,
                hipStream_t s) {
  TN_REQUIRE(m >= 1 && p >= 1 && m <= kMaxDimBig && p <= kMaxDimBig,
             "jacobi_svd: dimension out of range");
  if (batch <= 0) return;
  if (m > kMaxDim || p > kMaxDim) {
    // above the LDS-resident size: the matrix stays in global memory
    hipLaunchKernelGGL(jacobi_big_kernel, dim3(batch), dim3(1024), 0, s, W, m, p, tol,
                       max_sweeps, sigma, rot, nsteps);
    TN_HIP_CHECK(hipGetLastError());
    return;
  }
  const int pe = p + (p & 1);
  const size_t lds = (size_t)m * pe * sizeof(double);
  if (m == kMaxDim)
    hipLaunchKernelGGL((jacobi_kernel<true>), dim3(batch), dim3(1024), lds, s, W, m, p,
                       tol, max_sweeps, sigma, rot, nsteps);
  else
    hipLaunchKernelGGL((jacobi_kernel<false>), dim3(batch), dim3(1024), lds, s, W, m, p,
                       tol, max_sweeps, sigma, rot, nsteps);
  TN_HIP_CHECK(hipGetLastError());
}

void qrp(const double *A, int m, int n, double *W, double *Q, hipStream_t s) {
  TN_REQUIRE(m >= 1 && n >= 1 && m <= kMaxDim && n <= kMaxDim, "qrp: dimension out of range");
  const size_t lds = (size_t)m * (n | 1) * sizeof(double);
  hipLaunchKernelGGL(qrp_kernel, dim3(1), dim3(kQrpThreads), lds, s, A, m, n, W, Q);
  TN_HIP_CHECK(hipGetLastError());
}

void jacobi_accumulate(const double *rot, const int *nsteps, int p, double *J,
                       hipStream_t s, const double *J0, int rows) {
  TN_REQUIRE(p >= 1 && p <= kMaxDimBig, "jacobi_accumulate: p out of range");
  TN_REQUIRE(!J0 || (p <= kMaxDim && rows >= 1), "jacobi_accumulate: start matrix");
  if (p <= kMaxDim) {
    hipLaunchKernelGGL(jacobi_replay_kernel, dim3(J0 ? rows : p), dim3(64), 0, s, rot, nsteps, p,
                       J0, J);
  } else {
    // 2 rows per workgroup (timed on 128 x 128 replays, which this kernel
    // did before jacobi_replay_kernel: 286 us, 318 us with 4 rows, 394 us with 8)
    constexpr int ROWS = 2;
    hipLaunchKernelGGL((jacobi_accum_kernel<ROWS, kMaxDimBig>), dim3(ceil_div(p, ROWS)),
                       dim3(64), 0, s, rot, nsteps, p, J);
  }
  TN_HIP_CHECK(hipGetLastError());
}

void sort_desc(const double *sigma, int p, int batch, double *sorted,
               int *perm, hipStream_t s) {
  TN_REQUIRE(p <= kMaxDimBig, "sort_desc: p out of range");
  if (batch <= 0) return;
  hipLaunchKernelGGL(sort_desc_kernel, dim3(batch), dim3(128), 0, s, sigma, p,
                     batch, sorted, perm);
  TN_HIP_CHECK(hipGetLastError());
}

}  // namespace kern
}  // namespace tn
