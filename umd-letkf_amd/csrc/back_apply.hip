// back_apply.hip -- the transform of a group of many slabs for k < 64 without
// an eigensolve: M = sqrt(k-1) Tri^(-1/2) as a matrix, W = Q M Q^T from the
// stored reflectors, wbar = Q Tri^-1 Q^T b, and x_a = W x_b + wbar . x_b for
// every slab of the group (src/letkf_core.F90:100-141,
// src/letkf_solver.F90:284-290), all in FP64.
//
//  k_small_rational  the lower triangle of M from the two-term recurrences of
//                    the inverses (Tri + s_n I)^-1 (see kernels_transform.hip,
//                    k_mat_rational), one wave per problem, and Tri^-1 Q^T b;
//  k_back_apply      the two-sided back-transform and the apply with the
//                    matrix one row a lane, as tridiag_pair.h keeps it.
//
// wbar is A^-1 b and not W (W b) / (k-1): W is right to some units of 2^-53 of
// its largest entries, and b lies where W is smallest, so that the second form
// loses the square of the condition number (at 3e8, k = 50 with 12 slabs, the
// mean's increment was 9e-5 off, at 3e10 it was wrong; 4e-9 and 2e-7 so).
//
// They take the place of implicit QL with recorded rotations, the replay of
// the records into eigenvectors and two mat-vecs a slab (k_tql, k_replay,
// k_vec_apply, still run with LETKF_GPU_RAT=0): QL is a serial chain per
// problem, one lane each, and its records cross memory twice.  11 855
// problems of k = 40 with 50 slabs: 5.2 ms then, 0.51 ms now; 33 problems
// of k = 50 with 12 slabs: 540 us and 75 us.  The node table is the fine
// one (5e-16): over condition numbers of 1e2 to 8e6 the analysis is no further
// from the FP64 oracle than the eigensolve's (spread 2e-14 against 1e-13 at
// 8e6, k = 50).
#include <hip/hip_runtime.h>

#include "dpp_common.h"
#include "letkf_internal.h"

namespace lk {

constexpr int kGroupNodes = 16;   // nodes of one pass over the rows (18 KB of
                                  // LDS: eight waves a CU; all 62 would be two)

// Few problems or many, a wave's own latency is what this takes: the pivots'
// recurrence, and in the rows the reads of U (all lanes the same 16 values,
// two a read) and, from the second group of nodes on, of the entry to add to.
// Those are made a row and two rows ahead, and a row's multiplications run on
// the lanes below the diagonal alone instead of a select for each node: 342 ->
// 199 us at 11 855 problems of k = 40, 44 -> 24 us at 33 problems of k = 50.
__global__ __launch_bounds__(64) void k_small_rational(int k, int K, ChunkDev C,
                                                       double* __restrict__ B,
                                                       double* __restrict__ U,
                                                       const double* __restrict__ dd,
                                                       const double* __restrict__ ee, RatTab R) {
  constexpr int NG = kGroupNodes;
  constexpr int LD = NG + 2;        // 16-byte rows, lanes' own rows in different banks
  __shared__ double sd[66], se[66];
  // by row: U of the nodes' bottom-up pivots, and their top-down pivots; in the
  // two columns of Us that no node has, Q^T b and what its solve needs
  __shared__ __align__(16) double Us[66][LD], Gs[64][LD];
  const int64_t pair = blockIdx.x;
  if (!C.solve[pair]) return;
  const int l = threadIdx.x;
  double* Up = U + pair * K;
  const double m = (double)(k - 1);
  sd[l] = l < k ? dd[pair * K + l] : 0.0;
  se[l] = l < k - 1 ? ee[pair * K + l] : 0.0;
  Us[l][NG] = l < k ? Up[l] : 0.0;
  if (l < 2) { sd[64 + l] = 0.0; se[64 + l] = 0.0; Us[64 + l][NG] = 0.0; }
  __syncthreads();
  double gm = l < k ? sd[l] + (l > 0 ? fabs(se[l - 1]) : 0.0) + fabs(se[l]) : 0.0;
  gm = p_max<64>(gm);
  int bk = (int)ceil(log2(fmax(gm / m, 2.0)));
  bk = bk < 1 ? 1 : (bk > R.nb - 1 ? R.nb - 1 : bk);
  bk = __builtin_amdgcn_readfirstlane(bk);
  const int nn = __builtin_amdgcn_readfirstlane(R.n[bk]);
  const double* sn = R.tab + bk * kRatLd;
  const double* wn = sn + kRatLd / 2;
  double* Bp = B + pair * (int64_t)k * k;
  for (int n0 = 0; n0 < nn; n0 += NG) {
    // the pivots: lanes 0..15 top-down, lanes 16..31 bottom-up, a node each
    // (a node past the last has a pivot of at least m and weight 0).  Lane 32
    // goes with the first ones for Tri x = Q^T b: the pivots of Tri itself, and
    // the forward substitution by them.
    const bool sol = n0 == 0 && l == 2 * NG;
    if (l < 2 * NG || sol) {
      const int n = l & (NG - 1);
      const double sg = sol ? 0.0 : (n0 + n < nn ? m * sn[n0 + n] : m);
      double f = 0.0, e0 = 0.0;           // e0: the row before's off-diagonal
      if (l < NG || sol) {
        double d = sd[0], e1 = se[0], b = Us[0][NG], z = 0.0;
        double* out = sol ? &Us[0][NG] : &Gs[0][n];
        for (int i = 0; i < k; ++i) {
          const double d2 = sd[i + 1], e2 = se[i + 1], b2 = Us[i + 1][NG];
          const double D = fma(-e0, f, d + sg);
          const double ri = rcp_cubic(D);
          z = fma(-f, z, b);
          out[i * LD] = sol ? z * ri : D;
          f = e1 * ri;
          if (sol) Us[i][NG + 1] = f;
          e0 = e1;
          d = d2;
          e1 = e2;
          b = b2;
        }
      } else {
        double d = sd[k - 1], e1 = se[k - 2];
        for (int i = k - 1; i >= 0; --i) {
          const double d2 = sd[max(i - 1, 0)], e2 = se[max(i - 2, 0)];
          const double D = fma(-e0, f, d + sg);
          f = i > 0 ? e1 * rcp_cubic(D) : 0.0;
          Us[i][n] = f;
          e0 = e1;
          d = d2;
          e1 = e2;
        }
      }
    }
    __syncthreads();
    if (n0 == 0) {                        // x, entry l in lane l
      double x = 0.0, mine = 0.0;
#pragma unroll 4
      for (int i = k - 1; i >= 0; --i) {
        x = fma(-Us[i][NG + 1], x, Us[i][NG]);
        mine = l == i ? x : mine;
      }
      if (l < k) Up[l] = mine;
    }
    // the inverse's diagonal 1 / (D+_i + D-_i - (d_i + s)) = 1 / (D+_i - e_i U_(i+1)),
    // where column l starts
    double cf[NG], x[NG], u[NG];
    const int lr = l < k ? l : 0;
#pragma unroll
    for (int n = 0; n < NG; ++n) {
      cf[n] = n0 + n < nn ? m * wn[n0 + n] : 0.0;
      x[n] = rcp_cubic(fma(-se[lr], lr < k - 1 ? Us[lr + 1][n] : 0.0, Gs[lr][n]));
      u[n] = Us[0][n];
    }
    const bool more = n0 > 0 && l < k;
    auto old = [&](int r) { return more && r >= l && r < k ? Bp[r * k + l] : 0.0; };
    double o0 = old(0), o1 = old(1);
    // column l from its diagonal down
    for (int r = 0; r < k; ++r) {
      const double o2 = old(r + 2);
      double un[NG];
      const int rn = r + 1 < k ? r + 1 : r;
#pragma unroll
      for (int n = 0; n < NG; ++n) un[n] = Us[rn][n];
      if (r > l) {
#pragma unroll
        for (int n = 0; n < NG; ++n) x[n] = -u[n] * x[n];
      }
      double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int n = 0; n < NG; ++n) acc[n & 3] = fma(cf[n], x[n], acc[n & 3]);
      if (r >= l && l < k) Bp[r * k + l] = o0 + ((acc[0] + acc[1]) + (acc[2] + acc[3]));
      o0 = o1;
      o1 = o2;
#pragma unroll
      for (int n = 0; n < NG; ++n) u[n] = un[n];
    }
    __syncthreads();
  }
}

// P lanes a problem (two a wave for k <= 50), rows r and, with RPL = 2,
// r + 32.  The reflectors are walked backwards; reflector j has zeros up to
// entry j, so the blocks of 16 columns below it need no product and only the
// v_r w_c part of the update.  That is one loop for each block, not a branch
// in the step: the matrix stays in place in its registers (with the branch
// the compiler kept two copies of it and spilled).  x = Tri^-1 Q^T b rides along
// as row k, where v is zero: the product's row sum is v . x and the update
// x <- H x, so that the row ends as wbar.
template <int KQ, int P, int RPL>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
void k_back_apply(int k, int K, int64_t np, const int32_t* __restrict__ perm, LocDev L, StateDev S,
                  VarsDev V, ChunkDev C, DiagDev D, const double* __restrict__ B,
                  const double* __restrict__ U, const double* __restrict__ tau,
                  double* __restrict__ ana) {
  constexpr int NPW = 64 / P;
  constexpr int NT = (KQ + 15) / 16;
  __shared__ __align__(8) unsigned short sl[NPW][2048];
  const int lane = threadIdx.x;
  const int hh = P == 32 ? lane >> 5 : 0;
  const int r = lane & (P - 1), r1 = r + 32;
  const int64_t q = NPW * (int64_t)blockIdx.x + hh;
  int64_t pair = -1;
  if (q < np) pair = perm ? (int64_t)perm[q] : q;
  const bool act = pair >= 0 && C.solve[pair] != 0;
  if (__ballot(act) == 0ull) return;   // wave-uniform
  const int64_t pq = act ? pair : 0;
  const double* Bp = B + pq * (int64_t)k * k;
  const bool in0 = act && r < k, in1 = act && RPL == 2 && r1 < k;
  // the lane of row k (two rows a lane only for k >= 32)
  const bool bx = act && (RPL == 2 ? r1 : r) == k;
  const bool b0 = RPL == 1 && bx, b1 = RPL == 2 && bx;
  // every load is made, from an address inside the problem, and masked after
  const int rc = min(r, k - 1), rc1 = min(r1, k - 1);
  __shared__ double st[NPW][64];    // tau, then wbar
  for (int i = r; i < 64; i += P) st[hh][i] = act && i < k - 1 ? tau[pq * K + i] : 0.0;
  // M, symmetric, from its lower triangle (row-major in B), and row k from U:
  // chosen by the address (a lane that wrote over its row in a branch made the
  // compiler keep a second copy of the matrix, and spill)
  double a0[KQ], a1[RPL == 2 ? KQ : 1];
  const double* from0 = b0 ? U + pq * K : Bp;
  const double* from1 = b1 ? U + pq * K : Bp;
  const int d0 = b0 ? k : rc, o0 = b0 ? 0 : rc * k;      // entries up to the diagonal
  const int d1 = b1 ? k : rc1, o1 = b1 ? 0 : rc1 * k;
#pragma unroll
  for (int c = 0; c < KQ; ++c) {
    const int cc = min(c, k - 1);
    a0[c] = from0[cc <= d0 ? o0 + cc : cc * k + rc];
    if constexpr (RPL == 2) a1[c] = from1[cc <= d1 ? o1 + cc : cc * k + rc1];
    // bounds how many addresses are formed ahead
    if (c % 8 == 7) asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int c = 0; c < KQ; ++c) {
    a0[c] = (in0 || b0) && c < k ? a0[c] : 0.0;
    if constexpr (RPL == 2) a1[c] = (in1 || b1) && c < k ? a1[c] : 0.0;
  }
  __syncthreads();
  double n0 = 0.0, n1 = 0.0;
  auto fetch = [&](int j) __attribute__((always_inline)) {
    const double* row = Bp + max(j, 0) * k;
    n0 = row[rc];
    if constexpr (RPL == 2) n1 = row[rc1];
  };
  fetch(k - 2);
  // reflectors 16 B - 1 .. 16 B + 14 have zeros in the columns of blocks 0 .. B - 1
  static_for<NT>([&](auto I) __attribute__((always_inline)) {
    constexpr int blk = NT - 1 - decltype(I)::value;
    const int jlo = blk > 0 ? 16 * blk - 1 : 0;
    for (int j = min(k - 2, 16 * blk + 14); j >= jlo; --j) {
      // an unused reflector (t = 0) was not stored
      const double t = st[hh][j];
      const double v0 = in0 && r > j && t != 0.0 ? n0 : 0.0;
      double v1 = 0.0;
      if constexpr (RPL == 2) v1 = in1 && r1 > j && t != 0.0 ? n1 : 0.0;
      fetch(j - 1);
      double vq[4], p[4] = {0.0, 0.0, 0.0, 0.0};
      spread<P, RPL, NT>(v0, v1, vq);
      static_for<NT - blk>([&](auto T) __attribute__((always_inline)) {
        constexpr int tt = blk + decltype(T)::value;
        block_prod<KQ, RPL, tt>(p, vq[tt], a0, a1);
      });
      const double p0 = t * (p[0] + p[1]), p1 = t * (p[2] + p[3]);
      double pv = p0 * v0;
      if constexpr (RPL == 2) pv = fma(p1, v1, pv);
      const double kc = 0.5 * t * p_sum<P>(pv);
      const double w0 = fma(-kc, v0, p0), w1 = fma(-kc, v1, p1);
      double wq[4];
      spread<P, RPL, NT>(w0, w1, wq);
      static_for<NT>([&](auto T) __attribute__((always_inline)) {
        constexpr int tt = decltype(T)::value;
        block_upd<KQ, tt, (tt >= blk)>(a0, wq[tt], vq[tt], -v0, -w0);
        if constexpr (RPL == 2) block_upd<KQ, tt, (tt >= blk)>(a1, wq[tt], vq[tt], -v1, -w1);
      });
    }
  });
  // wbar, an entry a lane, added to every row: T = W + 1 wbar^T.  Every lane
  // writes its row, the others' where the slabs' list will be (a store in a
  // branch made the compiler spill).
  __syncthreads();
  {
    double* to = bx ? &st[hh][0] : reinterpret_cast<double*>(&sl[0][0]) + lane;
#pragma unroll
    for (int c = 0; c < KQ; ++c) to[c] = RPL == 2 ? a1[RPL == 2 ? c : 0] : a0[c];
  }
  __syncthreads();
  {
    double wq[4];
    spread<P, RPL, NT>(in0 ? st[hh][r] : 0.0, in1 ? st[hh][r1 & 63] : 0.0, wq);
    static_for<NT>([&](auto T) __attribute__((always_inline)) {
      constexpr int tt = decltype(T)::value;
      block_upd<KQ, tt, false>(a0, wq[tt], 0.0, 1.0, 0.0);
      if constexpr (RPL == 2) block_upd<KQ, tt, false>(a1, wq[tt], 0.0, 1.0, 0.0);
    });
  }
  auto mul = [&](double x0, double x1, double* o0, double* o1) __attribute__((always_inline)) {
    double xq[4], p[4] = {0.0, 0.0, 0.0, 0.0};
    spread<P, RPL, NT>(x0, x1, xq);
    static_for<NT>([&](auto T) __attribute__((always_inline)) {
      constexpr int tt = decltype(T)::value;
      block_prod<KQ, RPL, tt>(p, xq[tt], a0, a1);
    });
    *o0 = p[0] + p[1];
    *o1 = p[2] + p[3];
  };
  // slabs of each problem's group in ascending order
  const int64_t t_gp = pq / C.G;
  const int g = (int)(pq - t_gp * C.G);
  const int64_t ij = C.i0 + t_gp;
  const int mld = act ? D.mld[ij] : 0;
  int nsl = 0;
  for (int s0 = 0; s0 < S.ns; s0 += P) {
    const int s = s0 + r;
    const bool in = act && s < S.ns && slab_group(L, V, s, mld) == g;
    const unsigned long long bal = __ballot(in);
    const unsigned long long hb = P == 64 ? bal : (bal >> (32 * hh)) & 0xffffffffull;
    if (in) sl[hh][nsl + __popcll(hb & ((1ull << r) - 1ull))] = (unsigned short)s;
    nsl += __popcll(hb);
  }
  __syncthreads();
  int nmax = nsl;
  if constexpr (P == 32) nmax = max(nsl, __shfl_xor(nsl, 32, 64));
  nmax = __builtin_amdgcn_readfirstlane(nmax);
  const float* xb = S.state + (int64_t)S.k * S.ns * ij;
  double* xa = ana + (int64_t)S.k * S.ns * ij;
  auto slab = [&](int qs) { return (int64_t)k * (qs < nsl ? (int)sl[hh][qs] : 0); };
  int64_t so = slab(0);
  float x0 = (in0 && nsl > 0) ? xb[so + r] : 0.0f, x1 = (in1 && nsl > 0) ? xb[so + r1] : 0.0f;
  for (int qs = 0; qs < nmax; ++qs) {
    const int64_t sn = slab(qs + 1);
    const bool more = qs + 1 < nsl;
    const float y0 = (in0 && more) ? xb[sn + r] : 0.0f, y1 = (in1 && more) ? xb[sn + r1] : 0.0f;
    double o0, o1;
    mul((double)x0, (double)x1, &o0, &o1);
    if (qs < nsl) {
      if (in0) xa[so + r] = o0;
      if (in1) xa[so + r1] = o1;
    }
    so = sn;
    x0 = y0;
    x1 = y1;
  }
}

// the reduction has left T in dd and ee, the reflectors in B and tau and Q^T b in
// U (K entries a problem); perm: the order of the problems, nullptr for 0..np-1.
// Row k has to be one of a problem's rows: k = 32 takes two rows a lane.
void launch_back_apply(hipStream_t st, const LocDev& L, const StateDev& S, const VarsDev& V,
                       const ChunkDev& C, const DiagDev& D, double* B, double* U,
                       const double* tau, const double* dd, const double* ee, int K,
                       const RatTab& R, double* ana, const int32_t* perm) {
  const int64_t np = C.ngp * C.G;
  if (np <= 0) return;
  const int k = (int)S.k;
  k_small_rational<<<(unsigned)np, 64, 0, st>>>(k, K, C, B, U, dd, ee, R);
  const unsigned two = (unsigned)((np + 1) / 2);
#define LK_BACK(KQ, P, RPL, nb)                                                              \
  k_back_apply<KQ, P, RPL><<<nb, 64, 0, st>>>(k, K, np, perm, L, S, V, C, D, B, U, tau, ana)
  if (k <= 8) LK_BACK(8, 32, 1, two);
  else if (k <= 16) LK_BACK(16, 32, 1, two);
  else if (k <= 24) LK_BACK(24, 32, 1, two);
  else if (k <= 31) LK_BACK(32, 32, 1, two);
  else if (k <= 40) LK_BACK(40, 32, 2, two);
  else if (k <= 48) LK_BACK(48, 32, 2, two);
  else if (k <= 50) LK_BACK(50, 32, 2, two);
  else if (k <= 56) LK_BACK(56, 64, 1, (unsigned)np);
  else LK_BACK(64, 64, 1, (unsigned)np);
#undef LK_BACK
}

}  // namespace lk
