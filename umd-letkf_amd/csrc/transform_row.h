// transform_row.h -- the reduction and the back-transform of the explicit
// transform matrix (64 <= k <= 104, see transform_mat.h) with one row of the
// matrix in the registers of each lane, two waves a problem; the template,
// instantiated per row length KQ in transform_row_kq*.hip.
//
// A step takes v and w of every column to every lane by DPP (row_newbcast in
// v_fmac_f64, see tridiag_pair.h), so its multiplications are the matrix's
// own: 16 for a block of 16 columns in the product and 32 in the update.  The
// waves exchange the column, p = t A v and two sums through LDS, two barriers
// a step in the reduction and one in the back-transform, whose reflectors
// are known (its arrays are double buffered by step).  The blocks of columns
// that a reflector does not touch are left out by one loop for each first
// block (a branch in the step would make the compiler keep two copies of the
// matrix); the first wave leaves the reduction once its rows are reduced.
//
// A 2D grid of blocks (transform_blk.h) spends two instructions on other
// things for each multiplication: LDS reads of v and w for its rows and its
// columns, sums over the grid row, and the reflector's scalars in four waves
// with divisions and a root.  It still serves k > 104, whose rows do not fit
// the 256 registers of two waves a SIMD.
//
// Measured at 11 900 problems of k = 100: the reduction 4.3 ms as a 2D grid, 1.9
// this way, the back-transform 3.2 and 1.8.
//
//  k_row_tridiag<KQ>  A = Q Tri Q^T (LAPACK dsytd2, lower): reflector j in row
//                     j of B (columns > j), tau, d and e; Q^T b over b.
//  k_row_back<KQ>     W = Q M Q^T from M in the lower triangle of B, wbar from
//                     Tri^-1 Q^T b in b, and T = W + 1 wbar^T over B.
//
// b goes along an entry a lane, in LDS for the reduction, where a register
// more spills: its v . b is summed with v . p (wave_sums2).  As a row of the
// matrix, as tridiag_pair.h has it, it made rows of 88 and more spill.  The
// eigen stage of 11 952 problems at k = 64 / 80 / 100 / 104: 2.64 / 3.26 /
// 4.53 / 4.56 ms with W (W b) / (k - 1), which loses the square of the
// condition number, 2.71 / 3.35 / 4.58 / 4.74 ms now.
#pragma once

#include <hip/hip_runtime.h>

#include "dpp_common.h"
#include "letkf_internal.h"

namespace lk {

constexpr int kRowStride = 128;   // d, e, tau entries per problem (as kMatStride)

// a[C0 + e] of a wave-uniform e < 16
template <int KQ, int C0>
__device__ __forceinline__ double row_pick(const double (&a)[KQ], int e) {
  double x = a[C0];
#define LK_PICK(n) case n: if constexpr (C0 + n < KQ) x = a[C0 + n]; break;
  switch (e) {
    LK_PICK(1) LK_PICK(2) LK_PICK(3) LK_PICK(4) LK_PICK(5) LK_PICK(6) LK_PICK(7) LK_PICK(8)
    LK_PICK(9) LK_PICK(10) LK_PICK(11) LK_PICK(12) LK_PICK(13) LK_PICK(14) LK_PICK(15)
    default: break;
  }
#undef LK_PICK
  return x;
}

template <int KQ>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2)))
void k_row_tridiag(int k, ChunkDev C, double* __restrict__ B, double* __restrict__ bvec,
                   double* __restrict__ tau, double* __restrict__ dd, double* __restrict__ ee) {
  constexpr int NT = (KQ + 15) / 16;
  __shared__ double sx[128];        // column j of A below the diagonal
  __shared__ double sp[128];        // p = t A v
  __shared__ double ss[2], sd[2][2];   // the waves' sums of x . x; of v . p and v . b
  __shared__ double sb[128];        // b: an entry to the lane that holds the row
  const int64_t pair = blockIdx.x;
  if (!C.solve[pair]) return;
  const int r = threadIdx.x, lane = r & 63, i = r & 15;
  const int wv = __builtin_amdgcn_readfirstlane(r >> 6);
  double* Bp = B + pair * (int64_t)k * k;
  double* dp = dd + pair * kRowStride;
  double* ep = ee + pair * kRowStride;
  double* tp = tau + pair * kRowStride;
  // every load is made, from an address inside the problem, and masked after
  const int rc = min(r, k - 1);
  double a[KQ];
#pragma unroll
  for (int c = 0; c < KQ; ++c) a[c] = Bp[min(c, k - 1) * k + rc];
#pragma unroll
  for (int c = 0; c < KQ; ++c) {
    a[c] = r < k && c < k ? a[c] : 0.0;
    a[c] = r < k && c == r ? a[c] + (double)(k - 1) : a[c];
  }
  const double none[1] = {0.0};
  sb[r] = r < k ? bvec[pair * (int64_t)k + r] : 0.0;
  const int jend = k - 2;
  const int jl = wv == 0 ? min(64, jend) : jend;   // the wave's rows are reduced from here
  static_for<NT>([&](auto I) __attribute__((always_inline)) {
    constexpr int blk = decltype(I)::value;
    const int je = min(16 * blk + 16, jl);
    for (int j = 16 * blk; j < je; ++j) {
      const int j1 = j + 1;
      const double aj = row_pick<KQ, 16 * blk>(a, j - 16 * blk);
      if (r == j) dp[j] = aj;
      const double x = r > j ? aj : 0.0;
      sx[r] = x;
      const double xx = p_sum<64>(x * x);
      if (lane == 0) ss[wv] = xx;
      __syncthreads();
      double vq[NT], wq[NT];
#pragma unroll
      for (int t = blk; t < NT; ++t) vq[t] = sx[16 * t + i];
      const double alpha = sx[j1];
      const double s2 = ss[0] + ss[1];
      // a column of zeros (or below 1e-140 beside a diagonal of at least
      // k - 1): H_j = I; a NaN is not one
      const bool nz = !(s2 <= 1e-280);
      // 1 / mu and mu = sqrt(s2): the hardware estimate, two Newton steps,
      // one correction of the root
      double ri = __builtin_amdgcn_rsq(s2);
      ri = ri * fma(-0.5 * s2 * ri, ri, 1.5);
      ri = ri * fma(-0.5 * s2 * ri, ri, 1.5);
      double mu = s2 * ri;
      mu = fma(0.5 * ri, fma(-mu, mu, s2), mu);
      // beta = -sign(alpha) mu, v = x / (alpha - beta) with v_(j+1) = 1
      const double dab = fabs(alpha) + mu;
      const double t = nz ? dab * ri : 0.0;
      const double beta = nz ? -copysign(mu, alpha) : alpha;
      const double scal = nz ? copysign(rcp_cubic(dab), alpha) : 0.0;
      const double one = nz ? 1.0 : 0.0;
      const double v = r == j1 ? one : x * scal;
#pragma unroll
      for (int q = blk; q < NT; ++q) {
        vq[q] *= scal;
        if (q <= blk + 1) vq[q] = 16 * q + i == j1 ? one : vq[q];
      }
      double p[4] = {0.0, 0.0, 0.0, 0.0};
      static_for<NT - blk>([&](auto T) __attribute__((always_inline)) {
        constexpr int q = blk + decltype(T)::value;
        block_prod<KQ, 1, q>(p, vq[q], a, none);
      });
      const double pr = t * (p[0] + p[1]);
      sp[r] = pr;
      const double vp = wave_sums2(pr * v, v * sb[r]);
      if ((lane & 31) == 0) sd[lane >> 5][wv] = vp;
      // the reflector, and what only one row knows
      if (r > j && r < k) Bp[j * k + r] = v;
      if (r == j1) {
        tp[j] = t;
        ep[j] = beta;
      }
      __syncthreads();
      const double kc = 0.5 * t * (sd[0][0] + sd[0][1]);
      sb[r] = fma(-t * (sd[1][0] + sd[1][1]), v, sb[r]);
      const double w = fma(-kc, v, pr);
#pragma unroll
      for (int q = blk; q < NT; ++q) wq[q] = fma(-kc, vq[q], sp[16 * q + i]);
      static_for<NT - blk>([&](auto T) __attribute__((always_inline)) {
        constexpr int q = blk + decltype(T)::value;
        block_upd<KQ, q, true>(a, wq[q], vq[q], -v, -w);
      });
    }
  });
  // the first wave keeps the second's barriers; its sums are zero from here
  // (each is cleared where the second wave has read the last step's)
  if (jl < jend && lane == 0) ss[wv] = 0.0;
  for (int j = jl; j < jend; ++j) {
    __syncthreads();
    if (j == jl && (lane & 31) == 0) sd[lane >> 5][wv] = 0.0;
    __syncthreads();
  }
  // the last two diagonal entries and the last subdiagonal one
#pragma unroll
  for (int c = KQ > 10 ? KQ - 10 : 0; c < KQ; ++c) {
    if (c == k - 2) {
      if (r == k - 2) dp[k - 2] = a[c];
      if (r == k - 1) ep[k - 2] = a[c];
    }
    if (c == k - 1 && r == k - 1) dp[k - 1] = a[c];
  }
  if (r < k) bvec[pair * (int64_t)k + r] = sb[r];
}

template <int KQ>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2)))
void k_row_back(int k, ChunkDev C, double* __restrict__ B, double* bvec,
                const double* __restrict__ tau) {
  constexpr int NT = (KQ + 15) / 16;
  __shared__ double sv[2][128];     // the reflector of this step and of the next
  __shared__ double sp[2][128];     // p = t A v
  __shared__ double sd[2][2][2];    // the waves' sums of v . p and of v . x
  __shared__ double st[128];
  const int64_t pair = blockIdx.x;
  if (!C.solve[pair]) return;
  const int r = threadIdx.x, lane = r & 63, i = r & 15;
  const int wv = __builtin_amdgcn_readfirstlane(r >> 6);
  double* Bp = B + pair * (int64_t)k * k;
  const int rc = min(r, k - 1);
  const bool in = r < k;
  // M, symmetric, from its lower triangle (row-major in B)
  double a[KQ];
#pragma unroll
  for (int c = 0; c < KQ; ++c) {
    const int cc = min(c, k - 1);
    a[c] = Bp[max(rc, cc) * k + min(rc, cc)];
  }
  st[r] = r < k - 2 ? tau[pair * kRowStride + r] : 0.0;
  double x = in ? bvec[pair * (int64_t)k + r] : 0.0;   // Tri^-1 Q^T b, then wbar
  // v: reflector j's entry r; vn: the next step's, as loaded
  double v = in && r > k - 3 ? Bp[(k - 3) * k + rc] : 0.0;
  double vn = Bp[max(k - 4, 0) * k + rc];
  sv[(k - 3) & 1][r] = v;
#pragma unroll
  for (int c = 0; c < KQ; ++c) a[c] = in && c < k ? a[c] : 0.0;
  __syncthreads();
  const double none[1] = {0.0};
  // reflectors 16 B - 1 .. 16 B + 14 have zeros in the columns of blocks 0 .. B - 1
  static_for<NT>([&](auto I) __attribute__((always_inline)) {
    constexpr int blk = NT - 1 - decltype(I)::value;
    const int jlo = blk > 0 ? 16 * blk - 1 : 0;
    for (int j = min(k - 3, 16 * blk + 14); j >= jlo; --j) {
      const int buf = j & 1;
      const double t = st[j];
      double vq[NT], wq[NT];
#pragma unroll
      for (int q = blk; q < NT; ++q) vq[q] = sv[buf][16 * q + i];
      double p[4] = {0.0, 0.0, 0.0, 0.0};
      static_for<NT - blk>([&](auto T) __attribute__((always_inline)) {
        constexpr int q = blk + decltype(T)::value;
        block_prod<KQ, 1, q>(p, vq[q], a, none);
      });
      const double pr = t * (p[0] + p[1]);
      sp[buf][r] = pr;
      const double vp = wave_sums2(pr * v, v * x);
      if ((lane & 31) == 0) sd[buf][lane >> 5][wv] = vp;
      // the next reflector (the other buffer's readers, of step j + 1, have
      // passed that step's barrier), and the load of the one after it
      const double vx = in && r > j - 1 ? vn : 0.0;
      sv[buf ^ 1][r] = vx;
      vn = Bp[max(j - 2, 0) * k + rc];
      __syncthreads();
      const double kc = 0.5 * t * (sd[buf][0][0] + sd[buf][0][1]);
      x = fma(-t * (sd[buf][1][0] + sd[buf][1][1]), v, x);
      const double w = fma(-kc, v, pr);
#pragma unroll
      for (int q = 0; q < NT; ++q) {
        const double pc = sp[buf][16 * q + i];
        wq[q] = q >= blk ? fma(-kc, vq[q >= blk ? q : blk], pc) : pc;
      }
      static_for<NT>([&](auto T) __attribute__((always_inline)) {
        constexpr int q = decltype(T)::value;
        block_upd<KQ, q, (q >= blk)>(a, wq[q], vq[q >= blk ? q : blk], -v, -w);
      });
      v = vx;
    }
  });
  // wbar to memory and back: with x itself in the sums below the matrix's rows
  // spill (rows of 104: 0 -> 52 registers, 1.74 -> 1.84 ms at 11 952 problems)
  if (in) bvec[pair * (int64_t)k + r] = x;
  const double wb = in ? bvec[pair * (int64_t)k + r] : 0.0;
  // T = W + 1 wbar^T.  W is symmetric, so the lane that holds row r writes
  // column r, to which it adds wbar_r.
#pragma unroll
  for (int c = 0; c < KQ; ++c)
    if (in && c < k) Bp[c * k + r] = a[c] + wb;
}

template <int KQ>
void launch_row_tridiag_kq(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                           double* bvec, double* tau, double* dd, double* ee) {
  k_row_tridiag<KQ><<<nb, 128, 0, st>>>(k, C, B, bvec, tau, dd, ee);
}
template <int KQ>
void launch_row_back_kq(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                        double* bvec, const double* tau) {
  k_row_back<KQ><<<nb, 128, 0, st>>>(k, C, B, bvec, tau);
}

}  // namespace lk
