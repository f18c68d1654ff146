// tridiag_pair.h -- Householder tridiagonalization with the matrix in
// registers and every broadcast taken by DPP, two problems per wave (one for
// rows past 50); the template, instantiated per row length KQ in
// tridiag_pair_kq*.hip so that the fully unrolled kernels compile in
// parallel.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "eigen_common.h"
#include "letkf_internal.h"

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
// update with v = 0 and w = t v . x on that row is x <- H x.
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

template <typename F, int... I>
__device__ __forceinline__ void static_for_(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_(f, std::make_integer_sequence<int, N>{});
}

// the value of lane N of each 16-lane row
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x150 + N, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x150 + N, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// rows (0, 1, 2, 3) of 16 lanes -> e = (0, 0, 2, 2), o = (1, 1, 3, 3)
__device__ __forceinline__ void rows16(double v, double* e, double* o) {
  const unsigned l = (unsigned)__double2loint(v), h = (unsigned)__double2hiint(v);
  const auto sl = __builtin_amdgcn_permlane16_swap(l, l, false, false);
  const auto sh = __builtin_amdgcn_permlane16_swap(h, h, false, false);
  *e = __hiloint2double((int)sh[0], (int)sl[0]);
  *o = __hiloint2double((int)sh[1], (int)sl[1]);
}

// halves (0, 1) of the wave -> e = (0, 0), o = (1, 1)
__device__ __forceinline__ void rows32(double v, double* e, double* o) {
  const unsigned l = (unsigned)__double2loint(v), h = (unsigned)__double2hiint(v);
  const auto sl = __builtin_amdgcn_permlane32_swap(l, l, false, false);
  const auto sh = __builtin_amdgcn_permlane32_swap(h, h, false, false);
  *e = __hiloint2double((int)sh[0], (int)sl[0]);
  *o = __hiloint2double((int)sh[1], (int)sl[1]);
}

template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// sum over the P lanes of a problem, the same bits in every lane: rotations
// by 8, 4, 2 and 1 within the 16-lane rows (each stage adds the same two
// values in both lanes of a pair), then the rows' sums
template <int P>
__device__ __forceinline__ double p_sum(double x) {
  x += dpp_mov<0x128>(x);
  x += dpp_mov<0x124>(x);
  x += dpp_mov<0x122>(x);
  x += dpp_mov<0x121>(x);
  double e, o;
  rows16(x, &e, &o);
  x = e + o;
  if constexpr (P == 64) {
    rows32(x, &e, &o);
    x = e + o;
  }
  return x;
}

// largest value over the P lanes, in every lane
template <int P>
__device__ __forceinline__ double p_max(double x) {
  x = fmax(x, dpp_mov<0x128>(x));
  x = fmax(x, dpp_mov<0x124>(x));
  x = fmax(x, dpp_mov<0x122>(x));
  x = fmax(x, dpp_mov<0x121>(x));
  double e, o;
  rows16(x, &e, &o);
  x = fmax(e, o);
  if constexpr (P == 64) {
    rows32(x, &e, &o);
    x = fmax(e, o);
  }
  return x;
}

// q[t], t < NT: entry 16 t + i of a problem's vector in lane i of each of
// its 16-lane rows, from the lanes that own rows r (v0) and r + 32 (v1)
template <int P, int RPL, int NT>
__device__ __forceinline__ void spread(double v0, double v1, double (&q)[4]) {
  if constexpr (P == 32) {
    rows16(v0, &q[0], &q[1]);
    if constexpr (RPL == 2 && NT > 2) rows16(v1, &q[2], &q[3]);
  } else {
    double e, o;
    rows16(v0, &e, &o);
    rows32(e, &q[0], &q[2]);
    rows32(o, &q[1], &q[3]);
  }
}

// acc += q(lane N of the row) * x.  A VALU write of a register needs two
// wait states before DPP reads it, which the compiler does not see inside
// an asm statement: each one starts with them.
#define LK_FD(acc, q, x, n) \
  "v_fmac_f64_dpp " acc ", " q ", " x " row_newbcast:" n " row_mask:0xf bank_mask:0xf\n\t"
template <int N>
__device__ __forceinline__ void bfma(double& p, double q, double a) {
  asm("s_nop 1\n\t" LK_FD("%0", "%1", "%2", "%3") : "+&v"(p) : "v"(q), "v"(a), "n"(N));
}
template <int N>
__device__ __forceinline__ void bfma2(double& p0, double& p1, double q, double a0, double a1) {
  asm("s_nop 1\n\t" LK_FD("%0", "%2", "%3", "%5") LK_FD("%1", "%2", "%4", "%5")
      : "+&v"(p0), "+&v"(p1)
      : "v"(q), "v"(a0), "v"(a1), "n"(N));
}
// four columns N..N+3 of the product, two partial sums a row
template <int N>
__device__ __forceinline__ void bfma4(double& pa, double& pb, double q, double x0, double x1,
                                      double x2, double x3) {
  asm("s_nop 1\n\t" LK_FD("%0", "%2", "%3", "%7") LK_FD("%1", "%2", "%4", "%8")
      LK_FD("%0", "%2", "%5", "%9") LK_FD("%1", "%2", "%6", "%10")
      : "+&v"(pa), "+&v"(pb)
      : "v"(q), "v"(x0), "v"(x1), "v"(x2), "v"(x3), "n"(N), "n"(N + 1), "n"(N + 2), "n"(N + 3));
}
template <int N>
__device__ __forceinline__ void bfma42(double& p0a, double& p0b, double& p1a, double& p1b,
                                       double q, double x0, double x1, double x2, double x3,
                                       double y0, double y1, double y2, double y3) {
  asm("s_nop 1\n\t" LK_FD("%0", "%4", "%5", "%13") LK_FD("%2", "%4", "%9", "%13")
      LK_FD("%1", "%4", "%6", "%14") LK_FD("%3", "%4", "%10", "%14")
      LK_FD("%0", "%4", "%7", "%15") LK_FD("%2", "%4", "%11", "%15")
      LK_FD("%1", "%4", "%8", "%16") LK_FD("%3", "%4", "%12", "%16")
      : "+&v"(p0a), "+&v"(p0b), "+&v"(p1a), "+&v"(p1b)
      : "v"(q), "v"(x0), "v"(x1), "v"(x2), "v"(x3), "v"(y0), "v"(y1), "v"(y2), "v"(y3), "n"(N),
        "n"(N + 1), "n"(N + 2), "n"(N + 3));
}
// column N of the rank-2 update, a -= v_r w_c + w_r v_c (nv = -v_r, nw = -w_r)
template <int N>
__device__ __forceinline__ void upd(double& a, double wq, double vq, double nv, double nw) {
  asm("s_nop 1\n\t" LK_FD("%0", "%1", "%3", "%5") LK_FD("%0", "%2", "%4", "%5")
      : "+&v"(a)
      : "v"(wq), "v"(vq), "v"(nv), "v"(nw), "n"(N));
}
// four columns N..N+3 of it
template <int N>
__device__ __forceinline__ void upd4(double& a, double& b, double& c, double& d, double wq,
                                     double vq, double nv, double nw) {
  asm("s_nop 1\n\t" LK_FD("%0", "%4", "%6", "%8") LK_FD("%1", "%4", "%6", "%9")
      LK_FD("%2", "%4", "%6", "%10") LK_FD("%3", "%4", "%6", "%11")
      LK_FD("%0", "%5", "%7", "%8") LK_FD("%1", "%5", "%7", "%9")
      LK_FD("%2", "%5", "%7", "%10") LK_FD("%3", "%5", "%7", "%11")
      : "+&v"(a), "+&v"(b), "+&v"(c), "+&v"(d)
      : "v"(wq), "v"(vq), "v"(nv), "v"(nw), "n"(N), "n"(N + 1), "n"(N + 2), "n"(N + 3));
}
#undef LK_FD

// 1/x by the hardware estimate e0 and 1/x = e0 (1 + d + d^2 + ...), d = 1 -
// x e0 (at most 2^-22): cubic, so within rounding of a division.  The pivots
// of the rational solve are >= k - 1 > 0.
__device__ __forceinline__ double rcp_cubic(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double d = fma(-x, y, 1.0);
  return fma(y, fma(d, d, d), y);
}

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

// The rational solve of one problem per half (see k_tridiag_pair, RAT); all
// lanes of the wave take part (barrier, DPP sums), lanes of an inactive half
// or of a problem with more slabs than carried vectors store nothing.
// s_d, s_e and s_u hold T and the carried vectors of both halves, 0 past
// row k (1 on the diagonal).
template <int KQ, int NV>
__device__ __forceinline__ void rat_tail(int k, int K, bool act, int64_t pq, int nsl, int r,
                                         bool upper, const double* s_d, const double* s_e,
                                         const double* s_u, double* __restrict__ U,
                                         const double* __restrict__ rtab,
                                         const int* __restrict__ rtabn, int rnb) {
  constexpr int LDH = 66;
  const int hh = upper ? 1 : 0;
  const double* sdh = s_d + hh * LDH;
  const double* seh = s_e + hh * LDH;
  const bool valid = act && nsl <= NV - 1;
  // Gershgorin bound of the largest eigenvalue of T (SPD)
  double gm = 0.0;
#pragma unroll
  for (int i = r; i < KQ; i += 32)
    if (i < k) gm = fmax(gm, sdh[i] + (i > 0 ? fabs(seh[i - 1]) : 0.0) + fabs(seh[i]));
  gm = p_max<32>(gm);
  const double m = (double)(k - 1);
  const double kappa = gm / m;
  int b = (int)ceil(log2(fmax(kappa, 2.0)));
  b = b < 1 ? 1 : (b > rnb - 1 ? rnb - 1 : b);
  const int nn = rtabn[b];
  const bool node = r < 31;
  const double sigma = node ? (r < nn ? m * rtab[b * 64 + r] : m) : 0.0;
  const double coef = (node && r < nn) ? m * rtab[b * 64 + 32 + r] : 0.0;
  const int nv_h = valid ? nsl : 0;
  const int nsl_all = max(nv_h, __shfl_xor(nv_h, 32, 64));
  const int i0 = (int)(__brev((unsigned)r) >> 27);
  for (int q = 1; q <= nsl_all; ++q) {
    const bool actq = valid && q <= nsl;
    const double* ux = s_u + (hh * NV + (actq ? q : 0)) * LDH;
    const double* u = node ? ux : s_u + hh * NV * LDH;
    // LDL^T of T + sigma I with the forward substitution, then back; rows
    // past k are 1 on the diagonal and 0 elsewhere
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
    // lane 31: wbar . x_b = u_q . T^-1 u_b
    double wx = 0.0;
    if (!node) {
#pragma unroll
      for (int i = 0; i < KQ; ++i) {
        wx = fma(ux[i], p[i], wx);
        if ((i & 7) == 7) asm volatile("" ::: "memory");
      }
    }
    // y_i = sum over the node lanes of coef * x_i
#pragma unroll
    for (int i = 0; i < KQ; ++i) p[i] *= coef;
    __builtin_amdgcn_sched_barrier(0);
    half_sums_spread<KQ>(p, r);
    if (actq) {
      double* uo = U + (pq * NV + q) * K;
      if (i0 < k) uo[i0] = p[0];
      if constexpr (KQ > 32) {
        if (i0 + 32 < k) uo[i0 + 32] = p[1];
      }
      if (!node) uo[K - 1] = wx;
    }
  }
}

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
                    int* __restrict__ nvec, int* __restrict__ status,
                    const double* __restrict__ rtab, const int* __restrict__ rtabn, int rnb) {
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
    const int mld = act ? D.mld[ij] : 0;
    for (int s0 = 0; s0 < S.ns; s0 += P) {
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
      if constexpr (XS) {
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
      const double kc = 0.5 * t * p_sum<P>(pv);
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
    rat_tail<KQ, NV>(k, K, act, pq, nsl, r, upper, s_d, s_e, s_u, U, rtab, rtabn, rnb);
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
    if (NV > 0) nvec[pq] = nsl;
    status[pq] = NV > 0 && nsl > NV - 1 ? 3 : 0;   // more slabs than carried: Jacobi
  }
}

// one kernel of rows of KQ; returns 1 for the reduction alone, 2 with the
// rational solve
template <int KQ, int NV, int P, int RPL, bool XS>
int launch_tridiag_pair_nv(hipStream_t st, int64_t np, const int32_t* perm, int k, int K,
                           const LocDev& L, const StateDev& S, const VarsDev& V,
                           const ChunkDev& C, const DiagDev& D, double* B, const double* bvec,
                           double* tau, double* dd, double* ee, double* U, int* nvec,
                           int* status, const double* rtab, const int* rtabn, int rnb) {
  const unsigned nb = P == 32 ? (unsigned)((np + 1) / 2) : (unsigned)np;
  if constexpr (NV > 0 && P == 32) {
    if (rnb > 0) {
      k_tridiag_pair<KQ, NV, true, P, RPL, XS><<<nb, 64, 0, st>>>(
          k, K, np, perm, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, rtab, rtabn, rnb);
      return 2;
    }
  }
  k_tridiag_pair<KQ, NV, false, P, RPL, XS><<<nb, 64, 0, st>>>(
      k, K, np, perm, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, rtab, rtabn, rnb);
  return 1;
}

template <int KQ>
int launch_tridiag_pair_kq(hipStream_t st, int64_t np, const int32_t* perm, int NV, int k, int K,
                           const LocDev& L, const StateDev& S, const VarsDev& V,
                           const ChunkDev& C, const DiagDev& D, double* B, const double* bvec,
                           double* tau, double* dd, double* ee, double* U, int* nvec,
                           int* status, const double* rtab, const int* rtabn, int rnb) {
#define LK_GO(NV, P, RPL, XS)                                                               \
  return launch_tridiag_pair_nv<KQ, NV, P, RPL, XS>(st, np, perm, k, K, L, S, V, C, D, B, bvec, \
                                                    tau, dd, ee, U, nvec, status, rtab, rtabn, \
                                                    rnb)
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
    if (k + NV > 64) LK_NV(64, 1, true)
    LK_NV(64, 1, false)
  } else if constexpr (KQ > 32) {
    if (NV == 0) LK_GO(0, 32, 2, false);
    LK_NV(32, 2, false)   // k + NV <= 59
  } else {
    if (NV == 0) LK_GO(0, 32, 1, false);
    if (k + NV <= 32) LK_NV(32, 1, false)
    if constexpr (KQ > 16) LK_NV(32, 2, false)
    return 0;             // not reached: k + NV <= 16 + 9
  }
#undef LK_NV
#undef LK_GO
}

}  // namespace lk
