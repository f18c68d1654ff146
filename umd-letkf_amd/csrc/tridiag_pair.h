// tridiag_pair.h -- Householder tridiagonalization with the matrix in
// registers and every broadcast taken by DPP, two problems per wave (one for
// rows past 50); the template, instantiated per row length KQ in
// tridiag_pair_kq*.hip so that the fully unrolled kernels compile in
// parallel.
#pragma once

#include <hip/hip_runtime.h>

#include "dpp_common.h"
#include "eigen_common.h"
#include "letkf_internal.h"
#include "rat_solve.h"

namespace lk {

// ---------------------------------------------------------------------------
// P lanes reduce one problem (P = 32: one problem in each half of the wave;
// P = 64: one problem).  Lane r of the P keeps row r of A in a0[c] = A(r, c)
// and, with RPL = 2, row r + 32 in a1.  A step takes v_c and w_c of every
// column c to every lane.  Both are kept as vq[t], lane i of every 16-lane
// row holding entry 16 t + i (v_permlane16_swap / v_permlane32_swap of the
// lanes that own the entries), and v_fmac_f64 reads entry c as its first
// operand with row_newbcast:(c % 16), a DPP form that costs no more than
// the plain instruction.  So a step has no LDS traffic and no barrier: with
// v and w in LDS (16-byte broadcast reads, 40 a step) the LDS pipe, which
// eight waves of a CU share, was what bounded it.
//
// The vectors the transform needs (b = Yb^T R^-1 d and x_b of the group's
// slabs, NV of them) ride along as rows k .. k + NV - 1 of the matrix, rows
// that are there anyway: the product's row sum is v . x, and the rank-2
// update with v = 0 and w = t v . x on that row is x <- H x.  NV = 1: b alone
// (groups of many slabs, whose transform is formed as a matrix).
//
// A half past the end or on an unsolved problem computes on zeros and stores
// nothing; a step whose column is already reduced is a no-op by v = w =
// t = 0.  For steps j >= 31 of RPL = 2 the rows 0..31 are final and their
// updates are not compiled.  Rows at or above the pivot row are not masked:
// with v = 0 there, the update is a rotation of values that are not read.
//
// Measured at 620 000 problems of k = 50 with one carried slab (the
// 0.25-degree analysis, the rational solve included): 17.9 ms with
// v and w in LDS, 11.5 ms this way; 592 000 of k = 40 with two slabs 14.5 ms
// and 8.3 ms.
// ---------------------------------------------------------------------------

// RAT: the rational solve of the vector path runs in the same kernel after
// the reduction (P = 32 only), in the layout of k_ratsolve: lane j < 31 of
// a half solves (T + sigma_j I) x = Q^T x_b by LDL^T, lane 31 solves
// T x = Q^T b, and sums over the half form y = sqrt(k-1) T^(-1/2) Q^T x_b
// and wbar . x_b, written to U for k_qapply (T, Q^T b and the inputs stay
// on chip: no dd, ee or input U round trip, no separate launch).
//
// XS: the carried vectors are kept one entry a lane (xv) with a sum for each
// and step, for the ensembles whose problem has no rows to spare.
template <int KQ, int NV, bool RAT, int P, int RPL, bool XS>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
void k_tridiag_pair(int k, int K, int64_t np, const int32_t* __restrict__ perm, LocDev L,
                    StateDev S, VarsDev V, ChunkDev C, DiagDev D, double* __restrict__ B,
                    const double* __restrict__ bvec, double* __restrict__ tau,
                    double* __restrict__ dd, double* __restrict__ ee, double* __restrict__ U,
                    int* __restrict__ nvec, int* __restrict__ status, RatTab R) {
  static_assert(P == 32 || (P == 64 && RPL == 1 && !RAT), "");
  static_assert(!XS || (P == 64 && NV > 0), "");
  constexpr int NPW = 64 / P;             // problems per wave
  constexpr int LDH = 66;
  constexpr int NT = (KQ + 15) / 16;
  // rows 0..31 can hold carried vectors only where k can be below 32
  constexpr bool X0 = RPL == 1 || KQ <= 32;
  __shared__ int sl[NPW][NV > 0 ? NV : 1];
  __shared__ double s_u[NV > 0 ? NPW * NV * LDH : 1];
  __shared__ double s_d[RAT ? NPW * LDH : 1], s_e[RAT ? NPW * LDH : 1];
  const int lane = threadIdx.x;
  const bool upper = P == 32 && lane >= 32;
  const int hh = upper ? 1 : 0;
  const int r = lane & (P - 1), r1 = r + 32;
  const int64_t q = NPW * (int64_t)blockIdx.x + hh;
  int64_t pair = -1;
  if (q < np) pair = perm ? (int64_t)perm[q] : q;
  const bool act = pair >= 0 && C.solve[pair] != 0;
  if (__ballot(act) == 0ull) return;   // wave-uniform
  const int64_t pq = act ? pair : 0;
  const double* Bp = B + pq * (int64_t)k * k;
  double* Bw = B + pq * (int64_t)k * k;
  double a0[KQ], a1[RPL == 2 ? KQ : 1];
#pragma unroll
  for (int c = 0; c < KQ; ++c) {
    const double u0 = (act && r < k && c < k) ? Bp[r + (int64_t)k * c] : 0.0;
    a0[c] = (act && c == r && r < k) ? u0 + (double)(k - 1) : u0;
    if constexpr (RPL == 2) {
      const double u1 = (act && r1 < k && c < k) ? Bp[r1 + (int64_t)k * c] : 0.0;
      a1[c] = (act && c == r1 && r1 < k) ? u1 + (double)(k - 1) : u1;
    }
  }
  int nsl = 0;
  double xv[XS ? NV : 1];
  if constexpr (NV > 0) {
    // slabs of each problem's group in ascending order (ballot compaction
    // within its lanes)
    const int64_t t_gp = pq / C.G;
    const int g = (int)(pq - t_gp * C.G);
    const int64_t ij = C.i0 + t_gp;
    const int mld = act && NV > 1 ? D.mld[ij] : 0;
    for (int s0 = 0; NV > 1 && s0 < S.ns; s0 += P) {
      const int s = s0 + r;
      const bool in = act && s < S.ns && slab_group(L, V, s, mld) == g;
      const unsigned long long bal = __ballot(in);
      const unsigned long long hb = P == 64 ? bal : (bal >> (32 * hh)) & 0xffffffffull;
      const int qq = nsl + __popcll(hb & ((1ull << r) - 1ull));
      if (in && qq < NV - 1) sl[hh][qq] = s;
      nsl += __popcll(hb);
    }
    __syncthreads();
    double* su = s_u + hh * NV * LDH;
    const float* xb0 = S.state + (int64_t)S.k * S.ns * ij;
#pragma unroll
    for (int qv = 0; qv < NV; ++qv) {
      const bool have = act && (qv == 0 || qv <= nsl);
      const int64_t so = (have && qv > 0) ? (int64_t)k * sl[hh][qv > 0 ? qv - 1 : 0] : 0;
#pragma unroll
      for (int i = r; i < 64; i += P) {
        double x = 0.0;
        if (have && i < k) x = qv == 0 ? bvec[pq * (int64_t)k + i] : (double)xb0[so + i];
        su[qv * LDH + i] = x;
      }
    }
    __syncthreads();
    if constexpr (XS) {
#pragma unroll
      for (int qv = 0; qv < NV; ++qv) xv[qv] = su[qv * LDH + r];
    }
    // rows k .. k + NV - 1
    const int q0 = r - k, q1 = r1 - k;
    if (!XS && X0 && q0 >= 0 && q0 < NV) {
#pragma unroll
      for (int c = 0; c < KQ; ++c) a0[c] = su[q0 * LDH + c];
    }
    if constexpr (RPL == 2) {
      if (q1 >= 0 && q1 < NV) {
#pragma unroll
        for (int c = 0; c < KQ; ++c) a1[c] = su[q1 * LDH + c];
      }
    }
  }
  // tau and the off-diagonal of step j are kept by the lane of row j
  double t0 = 0.0, t1 = 0.0, e0 = 0.0, e1 = 0.0;
  static_for<KQ - 1>([&](auto J) __attribute__((always_inline)) {
    constexpr int j = decltype(J)::value;
    // static j: every a0[] / a1[] index below is a compile-time constant
    if (j <= k - 2) {
      constexpr bool lo_live = RPL == 1 || j < 31;   // rows 0..31 still have rows below j
      const double x0 = (lo_live && r > j && (!X0 || r < k)) ? a0[j] : 0.0;
      double x1 = 0.0;
      if constexpr (RPL == 2) x1 = (r1 > j && r1 < k) ? a1[j] : 0.0;
      double s2 = x0 * x0;
      if constexpr (RPL == 2) s2 = lo_live ? fma(x1, x1, s2) : x1 * x1;
      s2 = p_sum<P>(s2);
      double vq[4];
      spread<P, RPL, NT>(x0, x1, vq);
      const double alpha = row_bcast<(j + 1) & 15>(vq[(j + 1) >> 4]);
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
      const double v0 = lo_live ? (r == j + 1 ? one : x0 * scal) : 0.0;
      double v1 = 0.0;
      if constexpr (RPL == 2) v1 = (j + 1 >= 32 && r1 == j + 1) ? one : x1 * scal;
#pragma unroll
      for (int tt = (j + 1) >> 4; tt < NT; ++tt) {
        vq[tt] *= scal;
        if (tt == (j + 1) >> 4) vq[tt] = (lane & 15) == ((j + 1) & 15) ? one : vq[tt];
      }
      if constexpr (XS && NV > 3) {
        double dq[NV];
#pragma unroll
        for (int qv = 0; qv < NV; ++qv) dq[qv] = p_sum<P>(v0 * xv[qv]);
#pragma unroll
        for (int qv = 0; qv < NV; ++qv) xv[qv] = fma(-t * dq[qv], v0, xv[qv]);
      }
      // p = t A v over the columns right of j, and t v . x on the carried rows
      double p0a = 0.0, p0b = 0.0, p1a = 0.0, p1b = 0.0;
      constexpr int c4 = (j + 1 + 3) & ~3;   // the first aligned group of four
      static_for<(c4 < KQ ? c4 : KQ) - (j + 1)>([&](auto I) __attribute__((always_inline)) {
        constexpr int c = j + 1 + decltype(I)::value;
        if constexpr (RPL == 2 && lo_live) bfma2<c & 15>(p0a, p1a, vq[c >> 4], a0[c], a1[c]);
        else if constexpr (RPL == 2) bfma<c & 15>(p1a, vq[c >> 4], a1[c]);
        else bfma<c & 15>(p0a, vq[c >> 4], a0[c]);
      });
      static_for<(KQ > c4 ? (KQ - c4) / 4 : 0)>([&](auto I) __attribute__((always_inline)) {
        constexpr int c = c4 + 4 * decltype(I)::value;
        if constexpr (RPL == 2 && lo_live)
          bfma42<c & 15>(p0a, p0b, p1a, p1b, vq[c >> 4], a0[c], a0[c + 1], a0[c + 2], a0[c + 3],
                         a1[c], a1[c + 1], a1[c + 2], a1[c + 3]);
        else if constexpr (RPL == 2)
          bfma4<c & 15>(p1a, p1b, vq[c >> 4], a1[c], a1[c + 1], a1[c + 2], a1[c + 3]);
        else
          bfma4<c & 15>(p0a, p0b, vq[c >> 4], a0[c], a0[c + 1], a0[c + 2], a0[c + 3]);
      });
      constexpr int ct = KQ > c4 ? c4 + (KQ - c4) / 4 * 4 : KQ;   // rows of 50: two are left
      static_for<KQ - ct>([&](auto I) __attribute__((always_inline)) {
        constexpr int c = ct + decltype(I)::value;
        if constexpr (RPL == 2 && lo_live) bfma2<c & 15>(p0b, p1b, vq[c >> 4], a0[c], a1[c]);
        else if constexpr (RPL == 2) bfma<c & 15>(p1b, vq[c >> 4], a1[c]);
        else bfma<c & 15>(p0b, vq[c >> 4], a0[c]);
      });
      const double p0 = t * (p0a + p0b), p1 = t * (p1a + p1b);
      double pv = 0.0;
      if constexpr (lo_live) pv = p0 * v0;
      if constexpr (RPL == 2) pv = fma(p1, v1, pv);
      double kc;
      if constexpr (XS && NV <= 3) {
        // with the carried vectors' v . x: 2.79 -> 2.51 ms at 67 000 problems
        // of k = 63 with one slab
        double q[4] = {pv, v0 * xv[0], v0 * xv[1], NV > 2 ? v0 * xv[NV > 2 ? 2 : 0] : 0.0};
        wave_sums4(q);
        kc = 0.5 * t * q[0];
#pragma unroll
        for (int qv = 0; qv < NV; ++qv) xv[qv] = fma(-t * q[1 + qv], v0, xv[qv]);
      } else {
        kc = 0.5 * t * p_sum<P>(pv);
      }
      const double w0 = fma(-kc, v0, p0), w1 = fma(-kc, v1, p1);
      double wq[4];
      spread<P, RPL, NT>(w0, w1, wq);
      // rank-2 update A -= v w^T + w v^T on the columns right of j
      const double nv0 = -v0, nw0 = -w0, nv1 = -v1, nw1 = -w1;
      static_for<(c4 < KQ ? c4 : KQ) - (j + 1)>([&](auto I) __attribute__((always_inline)) {
        constexpr int c = j + 1 + decltype(I)::value;
        if constexpr (lo_live) upd<c & 15>(a0[c], wq[c >> 4], vq[c >> 4], nv0, nw0);
        if constexpr (RPL == 2) upd<c & 15>(a1[c], wq[c >> 4], vq[c >> 4], nv1, nw1);
      });
      static_for<(KQ > c4 ? (KQ - c4) / 4 : 0)>([&](auto I) __attribute__((always_inline)) {
        constexpr int c = c4 + 4 * decltype(I)::value;
        if constexpr (lo_live)
          upd4<c & 15>(a0[c], a0[c + 1], a0[c + 2], a0[c + 3], wq[c >> 4], vq[c >> 4], nv0, nw0);
        if constexpr (RPL == 2)
          upd4<c & 15>(a1[c], a1[c + 1], a1[c + 2], a1[c + 3], wq[c >> 4], vq[c >> 4], nv1, nw1);
      });
      static_for<KQ - ct>([&](auto I) __attribute__((always_inline)) {
        constexpr int c = ct + decltype(I)::value;
        if constexpr (lo_live) upd<c & 15>(a0[c], wq[c >> 4], vq[c >> 4], nv0, nw0);
        if constexpr (RPL == 2) upd<c & 15>(a1[c], wq[c >> 4], vq[c >> 4], nv1, nw1);
      });
      // reflector j, rows j+1..k-1
      if (lo_live && act && r > j && (!X0 || r < k)) Bw[(int64_t)j * k + r] = v0;
      if constexpr (RPL == 2) {
        if (act && r1 > j && r1 < k) Bw[(int64_t)j * k + r1] = v1;
      }
      if constexpr (j < 32 || P == 64) {
        t0 = r == j ? t : t0;
        e0 = r == j ? beta : e0;
      } else {
        t1 = r1 == j ? t : t1;
        e1 = r1 == j ? beta : e1;
      }
    }
    // keep the scheduler from interleaving steps (register pressure)
    __builtin_amdgcn_sched_barrier(0);
  });
  double dg0 = 0.0, dg1 = 0.0;
#pragma unroll
  for (int c = 0; c < KQ; ++c) {
    dg0 = (c == r) ? a0[c] : dg0;
    if constexpr (RPL == 2) dg1 = (c == r1) ? a1[c] : dg1;
  }
  // the carried vectors, Q^T b and Q^T x_b, are rows of the matrix still
  if constexpr (NV > 0) {
    double* su = s_u + hh * NV * LDH;
    if constexpr (XS) {
#pragma unroll
      for (int qv = 0; qv < NV; ++qv) su[qv * LDH + r] = r < k ? xv[qv] : 0.0;
    }
    const int q0 = r - k, q1 = r1 - k;
    if (!XS && X0 && q0 >= 0 && q0 < NV) {
#pragma unroll
      for (int c = 0; c < KQ; ++c) su[q0 * LDH + c] = c < k ? a0[c] : 0.0;
    }
    if constexpr (RPL == 2) {
      if (q1 >= 0 && q1 < NV) {
#pragma unroll
        for (int c = 0; c < KQ; ++c) su[q1 * LDH + c] = c < k ? a1[c] : 0.0;
      }
    }
  }
  if constexpr (RAT) {
    s_d[hh * LDH + r] = r < k ? dg0 : 1.0;
    s_e[hh * LDH + r] = r < k - 1 ? e0 : 0.0;
    s_d[hh * LDH + r1] = r1 < k ? dg1 : 1.0;
    s_e[hh * LDH + r1] = r1 < k - 1 ? e1 : 0.0;
    __syncthreads();
    const double* su = s_u + hh * NV * LDH;
    rat_vectors<KQ>(k, K, NV, act && nsl <= NV - 1, pq, nsl, r, s_d + hh * LDH, s_e + hh * LDH,
                    [su](int qv) { return su + qv * LDH; }, U, R);
  } else if constexpr (NV > 0) {
    __syncthreads();
  }
  if (!act) return;
  double* taup = tau + pq * K;
  double* ep = ee + pq * K;
  if (r < K) {
    taup[r] = r < k - 1 ? t0 : 0.0;
    if (!RAT) {
      dd[pq * K + r] = r < k ? dg0 : 0.0;
      ep[r] = r < k - 1 ? e0 : 0.0;
    }
  }
  if (P == 32 && r1 < K) {
    taup[r1] = r1 < k - 1 ? t1 : 0.0;
    if (!RAT) {
      dd[pq * K + r1] = r1 < k ? dg1 : 0.0;
      ep[r1] = r1 < k - 1 ? e1 : 0.0;
    }
  }
  if constexpr (NV > 0 && !RAT) {
    double* Up = U + pq * (int64_t)NV * K;
    const double* su = s_u + hh * NV * LDH;
#pragma unroll
    for (int qv = 0; qv < NV; ++qv)
#pragma unroll
      for (int i = r; i < 64; i += P)
        if (i < K) Up[qv * K + i] = i < k ? su[qv * LDH + i] : 0.0;
  }
  if (r == 0) {
    if (NV > 1) nvec[pq] = nsl;
    status[pq] = NV > 1 && nsl > NV - 1 ? 3 : 0;   // more slabs than carried: Jacobi
  }
}

// one kernel of rows of KQ; returns 1 for the reduction alone, 2 with the
// rational solve
template <int KQ, int NV, int P, int RPL, bool XS>
int launch_tridiag_pair_nv(hipStream_t st, int64_t np, const int32_t* perm, int k, int K,
                           const LocDev& L, const StateDev& S, const VarsDev& V,
                           const ChunkDev& C, const DiagDev& D, double* B, const double* bvec,
                           double* tau, double* dd, double* ee, double* U, int* nvec,
                           int* status, const RatTab& R) {
  const unsigned nb = P == 32 ? (unsigned)((np + 1) / 2) : (unsigned)np;
  if constexpr (NV > 1 && P == 32) {
    if (R.nb > 0) {
      k_tridiag_pair<KQ, NV, true, P, RPL, XS><<<nb, 64, 0, st>>>(
          k, K, np, perm, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
      return 2;
    }
  }
  k_tridiag_pair<KQ, NV, false, P, RPL, XS><<<nb, 64, 0, st>>>(
      k, K, np, perm, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
  return 1;
}

template <int KQ>
int launch_tridiag_pair_kq(hipStream_t st, int64_t np, const int32_t* perm, int NV, int k, int K,
                           const LocDev& L, const StateDev& S, const VarsDev& V,
                           const ChunkDev& C, const DiagDev& D, double* B, const double* bvec,
                           double* tau, double* dd, double* ee, double* U, int* nvec,
                           int* status, const RatTab& R) {
#define LK_GO(NV, P, RPL, XS)                                                               \
  return launch_tridiag_pair_nv<KQ, NV, P, RPL, XS>(st, np, perm, k, K, L, S, V, C, D, B, bvec, \
                                                    tau, dd, ee, U, nvec, status, R)
#define LK_NV(P, RPL, XS)          \
  switch (NV) {                    \
    case 2: LK_GO(2, P, RPL, XS);  \
    case 3: LK_GO(3, P, RPL, XS);  \
    case 5: LK_GO(5, P, RPL, XS);  \
    case 9: LK_GO(9, P, RPL, XS);  \
    default: return 0;             \
  }
  if constexpr (KQ > 50) {
    if (NV == 0) LK_GO(0, 64, 1, false);
    if (NV == 1) LK_GO(1, 64, 1, false);   // k <= 63
    if (k + NV > 64) LK_NV(64, 1, true)
    LK_NV(64, 1, false)
  } else if constexpr (KQ > 32) {
    if (NV == 0) LK_GO(0, 32, 2, false);
    if (NV == 1) LK_GO(1, 32, 2, false);
    LK_NV(32, 2, false)   // k + NV <= 59
  } else {
    if (NV == 0) LK_GO(0, 32, 1, false);
    if (NV == 1 && k < 32) LK_GO(1, 32, 1, false);
    if constexpr (KQ == 32) {
      if (NV == 1) LK_GO(1, 32, 2, false);
    }
    if (k + NV <= 32) LK_NV(32, 1, false)
    if constexpr (KQ > 16) LK_NV(32, 2, false)
    return 0;             // not reached: k + NV <= 16 + 9
  }
#undef LK_NV
#undef LK_GO
}

}  // namespace lk
