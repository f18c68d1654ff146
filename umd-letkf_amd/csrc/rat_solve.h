// rat_solve.h -- y = sqrt(k-1) T^(-1/2) u of a tridiagonal T by the rational
// approximation of x^(-1/2), two problems per wave (in the tridiagonalization
// of tridiag_pair.h, or k_ratsolve).
#pragma once

#include <hip/hip_runtime.h>

#include "dpp_common.h"
#include "letkf_internal.h"

namespace lk {

// One stage of the sums of p[0..n) over the lanes: lanes with `bit` go on
// with the odd entries, the others with the even ones, so n values of all
// lanes become (n + 1) / 2; CTRL brings the partner lane's value.
template <int CTRL, int N>
__device__ __forceinline__ void fold_stage(double (&p)[N], int n, bool bit) {
#pragma unroll
  for (int i = 0; i < N; i += 2) {
    if (i >= n) break;
    const double a = p[i], b = i + 1 < n ? p[i + 1] : 0.0;
    const double keep = bit ? b : a, send = bit ? a : b;
    p[i / 2] = keep + dpp_mov<CTRL>(send);
  }
}

// sums over each 32-lane half of p[0..KQ): entry 32 s + rev5(lane) is left
// in p[s] of lane `lane` (rev5: the five bits reversed).  3 to 7
// instructions a sum where one DPP sum chain for each takes 15.
template <int KQ>
__device__ __forceinline__ void half_sums_spread(double (&p)[KQ], int lane) {
#pragma unroll
  for (int i = 0; i < KQ; i += 2) {
    const double a = p[i], b = i + 1 < KQ ? p[i + 1] : 0.0;
    const auto l = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                    (unsigned)__double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                    (unsigned)__double2hiint(b), false, false);
    p[i / 2] = __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
  }
  constexpr int n1 = (KQ + 1) / 2, n2 = (n1 + 1) / 2, n3 = (n2 + 1) / 2, n4 = (n3 + 1) / 2;
  fold_stage<0x140>(p, n1, (lane & 8) != 0);   // row_mirror
  fold_stage<0x141>(p, n2, (lane & 4) != 0);   // row_half_mirror
  fold_stage<0x1b>(p, n3, (lane & 2) != 0);    // quad_perm 3 2 1 0
  fold_stage<0xb1>(p, n4, (lane & 1) != 0);    // quad_perm 1 0 3 2
}

// The node table's row for a problem and this lane's share of it.  The bound
// of the largest eigenvalue of T is Gershgorin's; T (sdh, seh) is in LDS, 1
// and 0 past row k.
struct RatRow {
  const double* s;   // nodes
  const double* w;   // weights
  int n;
  double m;
};
template <int KQ>
__device__ __forceinline__ RatRow rat_row(int k, int r, const double* sdh, const double* seh,
                                          const RatTab& R) {
  double gm = 0.0;
#pragma unroll
  for (int i = r; i < KQ; i += 32)
    if (i < k) gm = fmax(gm, sdh[i] + (i > 0 ? fabs(seh[i - 1]) : 0.0) + fabs(seh[i]));
  gm = p_max<32>(gm);
  const double m = (double)(k - 1);
  int b = (int)ceil(log2(fmax(gm / m, 2.0)));
  b = b < 1 ? 1 : (b > R.nb - 1 ? R.nb - 1 : b);
  const double* row = R.tab + b * kRatLd;
  return RatRow{row, row + kRatLd / 2, R.n[b], m};
}

// y = sqrt(k-1) T^(-1/2) u and wx = u . T^-1 ub of one problem in each half
// of a wave: lane j < 31 solves (T + sigma_j I) x = u by LDL^T, lane 31
// T x = ub, and the weighted sums of x over the lanes are y.  More than 31
// nodes take another round.  Entries r5 and r5 + 32 of y (r5: the lane's
// five bits reversed) come back in y0 and y1, wx in lane 31.  u and ub are
// in LDS, 0 past row k; every lane of the wave takes part.
template <int KQ>
__device__ __forceinline__ void rat_solve(int r, const RatRow& row, int rounds, const double* sdh,
                                          const double* seh, const double* u_slab,
                                          const double* u_b, double* y0, double* y1,
                                          double* wx_out) {
  const bool node = r < 31;
  const double* u = node ? u_slab : u_b;
  double s0 = 0.0, s1 = 0.0, wx = 0.0;
  for (int rd = 0; rd < rounds; ++rd) {
    const int j = 31 * rd + r;
    const bool on = node && j < row.n;
    const double sigma = node ? (on ? row.m * row.s[j] : row.m) : 0.0;
    const double coef = on ? row.m * row.w[j] : 0.0;
    double l[KQ], p[KQ];
    double rprev = 0.0, zprev = 0.0, eprev = 0.0;
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
      const double li = eprev * rprev;
      const double Di = fma(-li, eprev, sdh[i] + sigma);
      const double ri = rcp_cubic(Di);
      const double zi = fma(-li, zprev, u[i]);
      l[i] = li;
      p[i] = zi * ri;
      rprev = ri;
      zprev = zi;
      eprev = seh[i];
      // bounds how far the LDS reads are hoisted (their registers)
      if ((i & 7) == 7) asm volatile("" ::: "memory");
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = KQ - 2; i >= 0; --i) p[i] = fma(-l[i + 1], p[i + 1], p[i]);
    if (!node && rd == 0) {
#pragma unroll
      for (int i = 0; i < KQ; ++i) {
        wx = fma(u_slab[i], p[i], wx);
        if ((i & 7) == 7) asm volatile("" ::: "memory");
      }
    }
#pragma unroll
    for (int i = 0; i < KQ; ++i) p[i] *= coef;
    __builtin_amdgcn_sched_barrier(0);
    half_sums_spread<KQ>(p, r);
    s0 += p[0];
    if constexpr (KQ > 32) s1 += p[1];
  }
  *y0 = s0;
  *y1 = s1;
  *wx_out = wx;
}

// the solves of every slab of both halves' problems, into U (RAT below, and
// k_ratsolve); s_u(q) is the LDS vector q of this half
template <int KQ, typename VecOf>
__device__ __forceinline__ void rat_vectors(int k, int K, int NV, bool valid, int64_t pq, int nsl,
                                            int r, const double* sdh, const double* seh,
                                            VecOf&& vec, double* __restrict__ U,
                                            const RatTab& R) {
  const RatRow row = rat_row<KQ>(k, r, sdh, seh, R);
  const int mine = valid ? (row.n + 30) / 31 : 1;
  const int rounds = __builtin_amdgcn_readfirstlane(max(mine, __shfl_xor(mine, 32, 64)));
  const int nv_h = valid ? nsl : 0;
  const int nsl_all = __builtin_amdgcn_readfirstlane(max(nv_h, __shfl_xor(nv_h, 32, 64)));
  const int i0 = (int)(__brev((unsigned)r) >> 27);
  for (int q = 1; q <= nsl_all; ++q) {
    const bool actq = valid && q <= nsl;
    double y0, y1, wx;
    rat_solve<KQ>(r, row, rounds, sdh, seh, vec(actq ? q : 0), vec(0), &y0, &y1, &wx);
    if (actq) {
      double* uo = U + (pq * NV + q) * K;
      if (i0 < k) uo[i0] = y0;
      if constexpr (KQ > 32) {
        if (i0 + 32 < k) uo[i0 + 32] = y1;
      }
      if (r == 31) uo[K - 1] = wx;
    }
  }
}

}  // namespace lk
