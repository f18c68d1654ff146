// dpp_common.h -- broadcasts and sums by DPP and lane swaps, in FP64, of the
// kernels that keep a problem's matrix one row a lane (tridiag_pair.h,
// back_apply.hip, transform_row.h).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

namespace lk {

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
  if constexpr (P >= 32) {
    double e, o;
    rows16(x, &e, &o);
    x = e + o;
    if constexpr (P == 64) {
      rows32(x, &e, &o);
      x = e + o;
    }
  }
  return x;
}

// sums of four values over the wave, uniform: the halves' sums of two values
// take one swap and addition for both, so do the rows', and one chain of
// rotations serves the four rows that then hold a value each (29 instructions
// where four sums of their own take 104)
__device__ __forceinline__ double swap_sum32(double a, double b) {
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                  (unsigned)__double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                  (unsigned)__double2hiint(b), false, false);
  return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}
__device__ __forceinline__ double swap_sum16(double a, double b) {
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                  (unsigned)__double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                  (unsigned)__double2hiint(b), false, false);
  return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}
__device__ __forceinline__ void wave_sums4(double (&q)[4]) {
  // rows: q0, q2, q1, q3
  const double x = p_sum<16>(swap_sum16(swap_sum32(q[0], q[1]), swap_sum32(q[2], q[3])));
  const int lo = __double2loint(x), hi = __double2hiint(x);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = 16 * ((i & 1) * 2 + (i >> 1));
    q[i] = __hiloint2double(__builtin_amdgcn_readlane(hi, at), __builtin_amdgcn_readlane(lo, at));
  }
}

// sums of two values over the wave for the price of one: a's in lanes 0..31,
// b's in lanes 32..63
__device__ __forceinline__ double wave_sums2(double a, double b) {
  return p_sum<32>(swap_sum32(a, b));
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
// four columns of a -= v_r w_c alone
template <int N>
__device__ __forceinline__ void upd4v(double& a, double& b, double& c, double& d, double wq,
                                      double nv) {
  asm("s_nop 1\n\t" LK_FD("%0", "%4", "%5", "%6") LK_FD("%1", "%4", "%5", "%7")
      LK_FD("%2", "%4", "%5", "%8") LK_FD("%3", "%4", "%5", "%9")
      : "+&v"(a), "+&v"(b), "+&v"(c), "+&v"(d)
      : "v"(wq), "v"(nv), "n"(N), "n"(N + 1), "n"(N + 2), "n"(N + 3));
}
#undef LK_FD

// blocks of columns by 16: p += sum_c q(c) a[c], c = 16 T .. min(16 T + 15, KQ - 1)
template <int KQ, int RPL, int T>
__device__ __forceinline__ void block_prod(double (&p)[4], double q, const double (&a0)[KQ],
                                           const double (&a1)[RPL == 2 ? KQ : 1]) {
  constexpr int c0 = 16 * T, n = KQ - c0 < 16 ? KQ - c0 : 16;
  static_for<n / 4>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = 4 * decltype(I)::value, c = c0 + i;
    if constexpr (RPL == 2)
      bfma42<i>(p[0], p[1], p[2], p[3], q, a0[c], a0[c + 1], a0[c + 2], a0[c + 3], a1[c],
                a1[c + 1], a1[c + 2], a1[c + 3]);
    else
      bfma4<i>(p[0], p[1], q, a0[c], a0[c + 1], a0[c + 2], a0[c + 3]);
  });
  static_for<n % 4>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = n / 4 * 4 + decltype(I)::value, c = c0 + i;
    if constexpr (RPL == 2) bfma2<i>(p[0], p[2], q, a0[c], a1[c]);
    else bfma<i>(p[0], q, a0[c]);
  });
}

// a[c] -= v_r w_c (+ w_r v_c with VC) on one block of columns
template <int KQ, int T, bool VC>
__device__ __forceinline__ void block_upd(double (&a)[KQ], double wq, double vq, double nv,
                                          double nw) {
  constexpr int c0 = 16 * T, n = KQ - c0 < 16 ? KQ - c0 : 16;
  static_for<n / 4>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = 4 * decltype(I)::value, c = c0 + i;
    if constexpr (VC) upd4<i>(a[c], a[c + 1], a[c + 2], a[c + 3], wq, vq, nv, nw);
    else upd4v<i>(a[c], a[c + 1], a[c + 2], a[c + 3], wq, nv);
  });
  static_for<n % 4>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = n / 4 * 4 + decltype(I)::value, c = c0 + i;
    if constexpr (VC) upd<i>(a[c], wq, vq, nv, nw);
    else bfma<i>(a[c], wq, nv);
  });
}

// 1/x by the hardware estimate e0 and 1/x = e0 (1 + d + d^2 + ...), d = 1 -
// x e0 (at most 2^-22): cubic, so within rounding of a division.  The pivots
// of the rational solve are >= k - 1 > 0.
__device__ __forceinline__ double rcp_cubic(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double d = fma(-x, y, 1.0);
  return fma(y, fma(d, d, d), y);
}

}  // namespace lk
