// kernels_solve.hip -- the FP64 local transform and its application.
//
//   k_product_f64   Yb^T R^-1 Yb and Yb^T R^-1 d of one (gridpoint, group)
//                   on FP64 MFMA (v_mfma_f64_16x16x4f64)
//                   (src/letkf_core.F90:92-98,118-125)
//   k_eigen_apply   (k-1)I + Yb^T R^-1 Yb = V L V^T, T = V sqrt((k-1)/L) V^T
//                   + V L^-1 V^T Yb^T R^-1 d 1^T, x_a = x_b^T T for each slab of
//                   the group (src/letkf_core.F90:100-141,
//                   src/letkf_solver.F90:284-290)
//   k_finalize<NJ>  recenter, increment clip, RTPS, RTPP, multiplicative
//                   inflation, member bounds, spread
//                   (src/letkf_solver.F90:299-379)
#include <hip/hip_runtime.h>

#include <mutex>

#include <algorithm>

#include "dpp_common.h"
#include "eigen_common.h"
#include "letkf_internal.h"

namespace lk {

typedef double double4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// products: Yb^T R^-1 Yb and Yb^T R^-1 d of one (gridpoint, group) on FP64 MFMA
// (16x16x4), from the padded operand columns (hx in rows 0..k-1, the
// departure in row k, zeros above).  A wave keeps its 16x16 tiles of the
// upper triangle in registers and takes four observations a step: lane l
// holds row 16 b + l % 16 of observation l / 16 for every row block b its
// tiles touch, which is both MFMA operands' layout, so a step loads each
// value once, converts it once, and feeds NB (NB + 1) / 2 products of 64
// cycles from one run of loads.  Indices and scaled weights of 64 observations are
// read one lane each (one division an observation), a batch ahead, and
// passed on by lane shuffles; columns are loaded one step ahead.
//
// Up to k = 63 one wave holds all (at most 10) tiles: one wave a problem, or
// four that share its observations and add up through LDS where the chunk
// has too few problems to fill the chip (below 4096: 256 CUs x 4 SIMDs x 4
// waves).  Above, four waves share the tiles and each reads the columns its
// own tiles need.
//
// The kernel is bound by the matrix units: 5.5 ms at 160 600
// problems of k = 50 with 6.6e7 kept observations (4.6 ms at the rate of a
// large FP64 matrix product), where staging 64 converted observations in LDS
// for four waves, two LDS reads a product, took 18.9 ms.
// ---------------------------------------------------------------------------
constexpr int kFewProblems = 4096;

template <int NB>
__device__ constexpr int tile_row(int idx) {
  int r = 0;
  while (idx >= NB - r) { idx -= NB - r; ++r; }
  return r;
}
template <int NB>
__device__ constexpr int tile_col(int idx) {
  int r = 0;
  while (idx >= NB - r) { idx -= NB - r; ++r; }
  return r + idx;
}
// some tile of T0 .. T0 + N - 1 reads row block b
template <int NB, int T0, int N>
__device__ constexpr bool tile_reads(int b) {
  for (int i = T0; i < T0 + N; ++i)
    if (tile_row<NB>(i) == b || tile_col<NB>(i) == b) return true;
  return false;
}

// tiles T0 .. T0 + N - 1 over the observations ow, ow + OW, .. (in batches of 64)
template <int NB, int T0, int N, int OW>
__device__ __forceinline__ void product_tiles(const ObsDev& O, const int32_t* __restrict__ li,
                                              const float* __restrict__ lw, int64_t m, int ow,
                                              int lane, double4_t (&acc)[N]) {
  const int q = lane >> 4;
  // entry KT i + b of a column is row 16 b + i: a lane's rows are one run
  constexpr int KT = NB == 1 ? 1 : (NB + 1) & ~1;
  const float* __restrict__ col = O.hxp + KT * (lane & 15);
  const int64_t kp = O.kp;
  auto idx_at = [&](int64_t j) { return li[j + lane < m ? j + lane : 0]; };
  auto load = [&](int32_t id, float (&y)[NB]) __attribute__((always_inline)) {
    const float* c = col + (int64_t)id * kp;
    if constexpr (NB == 1) y[0] = *c;
    static_for<KT / 2>([&](auto I) __attribute__((always_inline)) {
      constexpr int b = 2 * decltype(I)::value;
      if constexpr (tile_reads<NB, T0, N>(b) || (b + 1 < NB && tile_reads<NB, T0, N>(b + 1))) {
        const float2 f = *(const float2*)(c + b);
        y[b] = f.x;
        if constexpr (b + 1 < NB) y[b + 1] = f.y;
      }
    });
  };
  int64_t j0 = 64 * (int64_t)ow;
  if (j0 >= m) return;
  // an entry past the list reads the list's first observation with weight 0
  int32_t idx = idx_at(j0);
  double sc = j0 + lane < m ? (double)lw[j0 + lane] / (double)O.err[idx] : 0.0;
  float y[NB] = {};
  load(__shfl(idx, q), y);
  for (; j0 < m; j0 += 64 * OW) {
    const int64_t jn = j0 + 64 * OW;
    const bool more = jn < m;
    const int32_t idx_n = more ? idx_at(jn) : idx;
    const bool on = jn + lane < m;
    const float w_n = on ? lw[jn + lane] : 0.0f;
    const float e_n = on ? O.err[idx_n] : 1.0f;
    const int nst = (int)min((int64_t)16, (m - j0 + 3) / 4);
#pragma unroll 2
    for (int st = 0; st < nst; ++st) {
      float yn[NB];
      const int nxt = 4 * (st + 1) + q;
      load(st + 1 < nst ? __shfl(idx, nxt) : __shfl(idx_n, q), yn);
      const double s = __shfl(sc, 4 * st + q);
      double u[NB], v[NB];
      static_for<NB>([&](auto I) __attribute__((always_inline)) {
        constexpr int b = decltype(I)::value;
        if constexpr (tile_reads<NB, T0, N>(b)) {
          u[b] = (double)y[b];
          v[b] = u[b] * s;
        }
      });
      static_for<N>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        constexpr int r = tile_row<NB>(T0 + i), c = tile_col<NB>(T0 + i);
        acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[r], u[c], acc[i], 0, 0, 0);
      });
      static_for<NB>([&](auto I) __attribute__((always_inline)) {
        constexpr int b = decltype(I)::value;
        if constexpr (tile_reads<NB, T0, N>(b)) y[b] = yn[b];
      });
    }
    idx = idx_n;
    sc = on ? (double)w_n / (double)e_n : 0.0;
  }
}

// register r of lane l of a tile: row 4r + l/16, column l%16; column k of the
// result is Yb^T R^-1 d.  A diagonal tile is complete, the others are mirrored.
template <int NB, int T0, int N>
__device__ __forceinline__ void product_store(const double4_t (&acc)[N], int k, int lane,
                                              double* __restrict__ Bp, double* __restrict__ bp) {
  static_for<N>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = decltype(I)::value;
    constexpr int tr = tile_row<NB>(T0 + i), tc = tile_col<NB>(T0 + i);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * tr + 4 * r + (lane >> 4);
      const int col = 16 * tc + (lane & 15);
      const double v = acc[i][r];
      if (row < k && col < k) {
        Bp[col + (int64_t)k * row] = v;
        if constexpr (tr != tc) Bp[row + (int64_t)k * col] = v;
      } else if (col == k && row < k) {
        bp[row] = v;
      }
    }
  });
}

// all tiles in one wave; OW waves share the observations
template <int NB, int OW>
__global__ __launch_bounds__(64 * OW) __attribute__((amdgpu_waves_per_eu(3)))
void k_product_f64(ObsDev O, int k, ChunkDev C, double* __restrict__ B,
                   double* __restrict__ bvec) {
  constexpr int N = NB * (NB + 1) / 2;
  __shared__ double red[OW > 1 ? 2 * N * 4 * 64 : 1];
  const int64_t pair = xcd_order(C.xcd, blockIdx.x, gridDim.x);
  if (!C.solve[pair]) return;
  const int64_t m = C.cnt[pair], off = C.off[pair];
  const int lane = threadIdx.x & 63;
  const int ow = OW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  double4_t acc[N];
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = (double4_t){0.0, 0.0, 0.0, 0.0};
  product_tiles<NB, 0, N, OW>(O, C.list_idx + off, C.list_w + off, m, ow, lane, acc);
  if constexpr (OW == 4) {
    // waves 2 and 3 into 0 and 1, then 1 into 0
#pragma unroll
    for (int h = 2; h >= 1; h >>= 1) {
      if (ow >= h && ow < 2 * h) {
        double* to = red + (ow - h) * (N * 256);
#pragma unroll
        for (int i = 0; i < 4 * N; ++i) to[i * 64 + lane] = acc[i >> 2][i & 3];
      }
      __syncthreads();
      if (ow < h) {
        const double* from = red + ow * (N * 256);
#pragma unroll
        for (int i = 0; i < 4 * N; ++i) acc[i >> 2][i & 3] += from[i * 64 + lane];
      }
      __syncthreads();
    }
    if (ow != 0) return;
  }
  product_store<NB, 0, N>(acc, k, lane, B + pair * (int64_t)k * k, bvec + pair * (int64_t)k);
}

// four waves share the tiles (k >= 64)
template <int NB>
__global__ __launch_bounds__(256) void k_product_f64_wide(ObsDev O, int k, ChunkDev C,
                                                          double* __restrict__ B,
                                                          double* __restrict__ bvec) {
  constexpr int NBLK = NB * (NB + 1) / 2, PER = (NBLK + 3) / 4;
  const int64_t pair = xcd_order(C.xcd, blockIdx.x, gridDim.x);
  if (!C.solve[pair]) return;
  const int64_t m = C.cnt[pair], off = C.off[pair];
  const int lane = threadIdx.x & 63;
  const int tw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double* Bp = B + pair * (int64_t)k * k;
  double* bp = bvec + pair * (int64_t)k;
  static_for<4>([&](auto W) __attribute__((always_inline)) {
    constexpr int w = decltype(W)::value;
    constexpr int T0 = w * PER, N = NBLK - T0 < PER ? NBLK - T0 : PER;
    if (tw == w) {
      double4_t acc[N];
#pragma unroll
      for (int i = 0; i < N; ++i) acc[i] = (double4_t){0.0, 0.0, 0.0, 0.0};
      product_tiles<NB, T0, N, 1>(O, C.list_idx + off, C.list_w + off, m, 0, lane, acc);
      product_store<NB, T0, N>(acc, k, lane, Bp, bp);
    }
  });
}

void launch_product_f64(hipStream_t st, const ObsDev& O, const StateDev& S,
                        const ChunkDev& C, double* B, double* bvec) {
  const int64_t np = C.ngp * C.G;
  if (np <= 0) return;
  const int k = (int)S.k;
  const unsigned nb = (unsigned)np;
  const bool few = np < kFewProblems;
#define LK_PROD(NB)                                               \
  if (few) k_product_f64<NB, 4><<<nb, 256, 0, st>>>(O, k, C, B, bvec); \
  else k_product_f64<NB, 1><<<nb, 64, 0, st>>>(O, k, C, B, bvec);      \
  break
  switch ((k + 1 + 15) / 16) {
    case 1: LK_PROD(1);
    case 2: LK_PROD(2);
    case 3: LK_PROD(3);
    case 4: LK_PROD(4);
    case 5: k_product_f64_wide<5><<<nb, 256, 0, st>>>(O, k, C, B, bvec); break;
    case 6: k_product_f64_wide<6><<<nb, 256, 0, st>>>(O, k, C, B, bvec); break;
    case 7: k_product_f64_wide<7><<<nb, 256, 0, st>>>(O, k, C, B, bvec); break;
    default: k_product_f64_wide<8><<<nb, 256, 0, st>>>(O, k, C, B, bvec); break;
  }
#undef LK_PROD
}

// ---------------------------------------------------------------------------
// eigensolve (parallel cyclic Jacobi, round-robin pair ordering) and the
// transform, one workgroup per (gridpoint, group); A and V live in LDS.
// ---------------------------------------------------------------------------
struct Rot { double c, s; int p, q; };

__device__ __forceinline__ void rr_pair(int n, int r, int i, int* p, int* q) {
  // round r of a round-robin tournament over n (even) players
  int a, b;
  if (i == 0) { a = 0; b = (r % (n - 1)) + 1; }
  else { a = ((r + i) % (n - 1)) + 1; b = ((r - i + (n - 1)) % (n - 1)) + 1; }
  *p = a < b ? a : b;
  *q = a < b ? b : a;
}

__global__ __launch_bounds__(256) void k_eigen_apply(LocDev L, StateDev S,
                                                     VarsDev V, ChunkDev C,
                                                     DiagDev D,
                                                     const double* __restrict__ B,
                                                     const double* __restrict__ bvec,
                                                     const int* __restrict__ only_flagged,
                                                     double* __restrict__ ana) {
  extern __shared__ double lds[];
  const int k = (int)S.k;
  const int n = (k + 1) & ~1;               // even number of players
  const int lda = n + 1;
  double* A = lds;                           // n x lda
  double* Vm = A + n * lda;                  // n x lda
  double* lam = Vm + n * lda;                // kMaxK
  double* u = lam + kMaxK;                   // kMaxK
  double* bb = u + kMaxK;                    // kMaxK
  double* fq = bb + kMaxK;                   // kMaxK
  Rot* rot = (Rot*)(fq + kMaxK);             // kMaxK / 2
  __shared__ int s_rot;
  __shared__ int s_nsl;
  __shared__ int s_sl[2048];

  // one block per problem, or, when only flagged problems are solved, a
  // bounded grid that strides over 256-problem runs of the chunk: one load
  // per thread finds whether a run holds a flagged problem, and the block
  // then walks that run's problems together, so the barriers below stay
  // uniform
  const int64_t npair = C.ngp * C.G;
  const int64_t rstep = only_flagged ? (int64_t)gridDim.x * 256 : (int64_t)gridDim.x;
  for (int64_t rbase = only_flagged ? (int64_t)blockIdx.x * 256 : (int64_t)blockIdx.x;
       rbase < npair; rbase += rstep) {
  int64_t rend = rbase + 1;
  if (only_flagged) {
    const int64_t mine = rbase + threadIdx.x;
    const int fl = (mine < npair && C.solve[mine] && only_flagged[mine] != 0) ? 1 : 0;
    if (!__syncthreads_or(fl)) continue;
    rend = rbase + 256 < npair ? rbase + 256 : npair;
  }
  for (int64_t pair = rbase; pair < rend; ++pair) {
  if (!C.solve[pair]) continue;
  if (only_flagged && only_flagged[pair] == 0) continue;
  const int tid = threadIdx.x;
  const int64_t t = pair / C.G;
  const int g = (int)(pair - t * C.G);
  const int64_t ij = C.i0 + t;
  const double* Bp = B + pair * (int64_t)k * k;

  for (int e = tid; e < n * n; e += 256) {
    const int i = e / n, j = e - i * n;
    double v = 0.0;
    // upper triangle only: the tridiagonalization overwrites the lower one
    if (i < k && j < k) v = i <= j ? Bp[i + (int64_t)k * j] : Bp[j + (int64_t)k * i];
    if (i == j) v += (i < k) ? (double)(k - 1) : 1.0;   // dummy player: isolated 1
    A[i * lda + j] = v;
    Vm[i * lda + j] = (i == j) ? 1.0 : 0.0;
  }
  for (int i = tid; i < k; i += 256) bb[i] = bvec[pair * (int64_t)k + i];
  __syncthreads();

  const int half = n / 2;
  for (int sweep = 0; sweep < 40; ++sweep) {
    if (tid == 0) s_rot = 0;
    __syncthreads();
    for (int r = 0; r < n - 1; ++r) {
      if (tid < half) {
        int p, q;
        rr_pair(n, r, tid, &p, &q);
        double c = 1.0, s = 0.0;
        if (q < k) {
          const double apq = A[p * lda + q];
          const double app = A[p * lda + p], aqq = A[q * lda + q];
          if (apq != 0.0 && fabs(apq) > 1e-18 * sqrt(fabs(app) * fabs(aqq))) {
            const double tau = (aqq - app) / (2.0 * apq);
            double tt;
            if (fabs(tau) > 1e150) tt = 0.5 / tau;
            else tt = (tau >= 0.0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
            c = 1.0 / sqrt(1.0 + tt * tt);
            s = tt * c;
            s_rot = 1;
          }
        }
        rot[tid] = Rot{c, s, p, q};
      }
      __syncthreads();
      for (int e = tid; e < half * n; e += 256) {       // rows p, q of A
        const int i = e / n, col = e - i * n;
        const Rot R = rot[i];
        if (R.s != 0.0) {
          const double apk = A[R.p * lda + col], aqk = A[R.q * lda + col];
          A[R.p * lda + col] = R.c * apk - R.s * aqk;
          A[R.q * lda + col] = R.s * apk + R.c * aqk;
        }
      }
      __syncthreads();
      for (int e = tid; e < half * n; e += 256) {       // columns p, q of A, V
        const int i = e / n, row = e - i * n;
        const Rot R = rot[i];
        if (R.s != 0.0) {
          const double akp = A[row * lda + R.p], akq = A[row * lda + R.q];
          A[row * lda + R.p] = R.c * akp - R.s * akq;
          A[row * lda + R.q] = R.s * akp + R.c * akq;
          const double vkp = Vm[row * lda + R.p], vkq = Vm[row * lda + R.q];
          Vm[row * lda + R.p] = R.c * vkp - R.s * vkq;
          Vm[row * lda + R.q] = R.s * vkp + R.c * vkq;
        }
      }
      __syncthreads();
      if (tid < half) {
        const Rot R = rot[tid];
        if (R.s != 0.0) { A[R.p * lda + R.q] = 0.0; A[R.q * lda + R.p] = 0.0; }
      }
      __syncthreads();
    }
    if (s_rot == 0) break;
    __syncthreads();
  }

  // T = V diag(sqrt((k-1)/lam)) V^T + wbar 1^T,  wbar = V diag(1/lam) V^T b
  for (int i = tid; i < k; i += 256) {
    lam[i] = A[i * lda + i];
    fq[i] = sqrt((double)(k - 1) / lam[i]);
  }
  __syncthreads();
  for (int i = tid; i < k; i += 256) {
    double acc = 0.0;
    for (int a = 0; a < k; ++a) acc += Vm[a * lda + i] * bb[a];
    u[i] = acc / lam[i];
  }
  __syncthreads();
  for (int a = tid; a < k; a += 256) {
    double acc = 0.0;
    for (int i = 0; i < k; ++i) acc += Vm[a * lda + i] * u[i];
    bb[a] = acc;                               // wbar
  }
  __syncthreads();
  for (int e = tid; e < k * k; e += 256) {
    const int a = e / k, c = e - a * k;
    double acc = 0.0;
    for (int i = 0; i < k; ++i) acc += Vm[a * lda + i] * fq[i] * Vm[c * lda + i];
    A[a * lda + c] = acc + bb[a];              // T(a, c)
  }
  if (tid == 0) {
    int nsl = 0;
    const int mld = D.mld[ij];
    for (int s = 0; s < S.ns && nsl < 2048; ++s)
      if (slab_group(L, V, s, mld) == g) s_sl[nsl++] = s;
    s_nsl = nsl;
  }
  __syncthreads();
  const int nsl = s_nsl;
  const float* xb0 = S.state + (int64_t)S.k * S.ns * ij;
  double* xa0 = ana + (int64_t)S.k * S.ns * ij;
  for (int e = tid; e < nsl * k; e += 256) {   // x_a = x_b^T T
    const int sl = s_sl[e / k], j = e % k;
    const float* xb = xb0 + (int64_t)k * sl;
    double acc = 0.0;
    for (int i = 0; i < k; ++i) acc += (double)xb[i] * A[i * lda + j];
    xa0[(int64_t)k * sl + j] = acc;
  }
  __syncthreads();                            // LDS reused by the next problem
  }
  }
}

size_t eigen_lds_bytes(int k) {
  const int n = (k + 1) & ~1;
  return sizeof(double) * (2 * (size_t)n * (n + 1) + 4 * kMaxK) + sizeof(Rot) * (kMaxK / 2 + 1);
}

hipError_t launch_eigen_apply_f64(hipStream_t st, const LocDev& L, const StateDev& S,
                                  const VarsDev& V, const ChunkDev& C,
                                  const DiagDev& D, const double* B,
                                  const double* bvec, const int* only_flagged, double* ana) {
  const int64_t np = C.ngp * C.G;
  if (np <= 0) return hipSuccess;
  const size_t lds = eigen_lds_bytes((int)S.k);
  // the dynamic LDS limit is raised once per process, thread-safely; its
  // result is kept and returned by every later launch
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [] {
    attr_err = hipFuncSetAttribute((const void*)k_eigen_apply,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
  });
  if (attr_err != hipSuccess) return attr_err;
  const unsigned nb = only_flagged ? (unsigned)std::min<int64_t>(np, 1024) : (unsigned)np;
  k_eigen_apply<<<nb, 256, lds, st>>>(L, S, V, C, D, B, bvec, only_flagged, ana);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// post-processing.  Every step of src/letkf_solver.F90:299-379 acts slab by
// slab, and the slabs of all gridpoints follow one another: a wave takes four
// at a time, one in each of its 16-lane rows with members i + 16 j in lane i.
// A sum is NJ - 1 additions and four DPP rotations, and the roots and
// divisions serve four slabs (with one slab a wave, 250 instructions each,
// the instructions bounded it: 684 us at 1.04e6 slabs of k = 50, 397 us at
// 810 000 of k = 40, against 150 and 80 us of memory traffic; now 279 and
// 173 us).  Small grids: one slab's latency instead of a gridpoint's slabs
// in turn.
//
// A run of slabs is looked over first, a lane each: which are solved,
// masked (the background unchanged) or, with skip_solved, done already by
// the apply.  A run is the four slabs of one pass, or 16 where the apply has
// done most of them and the waves' launch counts (972 000 slabs of k = 100, 30%
// of them masked: 131 us with four, 104 with 16, 79 with masked slabs copied
// without the sums).
// ---------------------------------------------------------------------------
template <int NJ>
__global__ __launch_bounds__(256) void k_finalize(LocDev L, StateDev S, VarsDev V, ChunkDev C,
                                                  DiagDev D, float rtps, float rtpp, float mul,
                                                  double* __restrict__ ana,
                                                  double* __restrict__ amean,
                                                  double* __restrict__ asprd, bool skip_solved,
                                                  uint32_t n, int run) {
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t u64 = ((int64_t)blockIdx.x * 4 + wid) * run;
  if (u64 >= n) return;
  const uint32_t u0 = (uint32_t)u64;
  const int k = (int)S.k;
  int s_own = 0;
  bool solved = false, masked = false, need = false;
  if (lane < run && u0 + lane < n) {
    const uint32_t t = (u0 + lane) / (uint32_t)S.ns;
    s_own = (int)(u0 + lane - t * (uint32_t)S.ns);
    const int64_t ij = C.i0 + t;
    masked = S.mask[ij] != 0;
    const int g = slab_group(L, V, s_own, D.mld[ij]);
    solved = !masked && g >= 0 && C.solve[(int64_t)t * C.G + g];
    need = !(skip_solved && solved);
  }
  const uint64_t b_solved = __ballot(solved), b_masked = __ballot(masked), b_need = __ballot(need);
  const double dk = (double)k, dk1 = (double)(k - 1);
  const int i = lane & 15;
  // passes of masked slabs alone are a copy, and out of the loop below, where
  // the copy cost every other pass 5% (1.04e6 slabs of k = 50 without masks 293 us;
  // 277 without the copy, 279 this way; 810 000 of k = 40, 30% masked: 184, 195 and
  // 173)
  uint64_t todo = b_need;
  for (int q = 0; q < run && (b_need & b_masked) != 0; q += 4) {
    const uint32_t nd = (uint32_t)(b_need >> q) & 15u, mk = (uint32_t)(b_masked >> q) & 15u;
    if (nd == 0 || (nd & ~mk) != 0) continue;         // wave-uniform
    todo &= ~(15ull << q);
    const int at = q + (lane >> 4);
    if (((b_need >> at) & 1) == 0) continue;
    const int64_t e = C.i0 * S.ns + u0 + at;
    const float* xb = S.state + e * k;
    double* xa = ana + e * k;
    float c[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) c[j] = xb[min(i + 16 * j, k - 1)];
    const float cm = S.mean[e], cs = S.sprd[e];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (i + 16 * j < k) xa[i + 16 * j] = (double)c[j];
    if (i == 0) {
      amean[e] = (double)cm;
      asprd[e] = (double)cs;
    }
  }
  for (int q = 0; q < run; q += 4) {
    if (((todo >> q) & 15) == 0) continue;            // wave-uniform
    const int at = q + (lane >> 4);
    const bool on = (todo >> at) & 1, sol = (b_solved >> at) & 1, msk = (b_masked >> at) & 1;
    const int s = __shfl(s_own, at, 64);
    const int64_t e = C.i0 * S.ns + u0 + at;          // slab of the whole grid
    const float* xb = S.state + e * k;
    double* xa = ana + e * k;
    double x[NJ];
    float b[NJ];
    if (on) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        b[j] = (!sol || rtpp > 0.0f) && i + 16 * j < k ? xb[i + 16 * j] : 0.0f;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        x[j] = sol && i + 16 * j < k ? xa[i + 16 * j] : (double)b[j];
    } else {
#pragma unroll
      for (int j = 0; j < NJ; ++j) { b[j] = 0.0f; x[j] = 0.0; }
    }
    const double bm = on ? (double)S.mean[e] : 0.0, bs = on ? (double)S.sprd[e] : 0.0;
    const int v = on ? V.slab_var[s] : -1;
    double blo = 0.0, bhi = 0.0, inc = 0.0;
    if (v >= 0) {
      inc = (double)V.inc_max[v];
      blo = (double)V.bounds[2 * v];
      bhi = (double)V.bounds[2 * v + 1];
    }
    auto sum = [&](auto f) __attribute__((always_inline)) {
      double p = 0.0;
#pragma unroll
      for (int j = 0; j < NJ; ++j) p += i + 16 * j < k ? f(x[j]) : 0.0;
      return p_sum<16>(p);
    };
    auto self = [](double y) { return y; };
    auto sq = [](double y) { return y * y; };
    // recenter (:299-303)
#pragma unroll
    for (int j = 0; j < NJ; ++j) x[j] += bm;
    double mean = sum(self) / dk;
#pragma unroll
    for (int j = 0; j < NJ; ++j) x[j] -= mean;
    // increment clipping (:308-318)
    if (v >= 0) {
      double r = mean - bm;
      r = fmax(r, -inc);
      r = fmin(r, inc);
      r = fmax(r, blo - bm);
      r = fmin(r, bhi - bm);
      mean = r + bm;
    }
    // RTPS (:322-335)
    if (rtps > 0.0f) {
      const double sa = sqrt(sum(sq) / dk1);
      const double f = sa > 0.0 ? (double)rtps * (bs - sa) / sa + 1.0 : 1.0;
#pragma unroll
      for (int j = 0; j < NJ; ++j) x[j] *= f;
    }
    // RTPP (:339-343)
    if (rtpp > 0.0f) {
      const double a = (double)rtpp;
#pragma unroll
      for (int j = 0; j < NJ; ++j) x[j] = a * (double)b[j] + (1.0 - a) * x[j];
    }
    // multiplicative (:347-349)
    if (mul != 1.0f) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) x[j] *= (double)mul;
    }
    // member bounds and re-mean (:357-371)
    if (__ballot(v >= 0)) {
      if (v >= 0) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) x[j] = fmin(fmax(x[j], blo - mean), bhi - mean);
      }
      const double r = sum(self) / dk;
      if (v >= 0) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) x[j] -= r;
        mean += r;
      }
    }
    // final spread and members (:375-379)
    const double sp = sqrt(sum(sq) / dk1);
    if (on) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (i + 16 * j < k) xa[i + 16 * j] = msk ? (double)b[j] : x[j] + mean;
      if (i == 0) {
        amean[e] = msk ? bm : mean;
        asprd[e] = msk ? bs : sp;
      }
    }
  }
}

void launch_finalize(hipStream_t st, const LocDev& L, const StateDev& S,
                     const VarsDev& V, const ChunkDev& C, const DiagDev& D,
                     const FinArgs& F, double* ana, bool skip_solved) {
  // slabs are numbered in 32 bits: gridpoints in parts of at most 2^31 slabs
  const int64_t part = std::max<int64_t>(1, (1ll << 31) / std::max<int64_t>(S.ns, 1) - 1);
  for (int64_t t0 = 0; t0 < C.ngp && S.ns > 0; t0 += part) {
    ChunkDev P = C;
    P.i0 = C.i0 + t0;
    P.ngp = std::min(part, C.ngp - t0);
    P.solve = C.solve + t0 * C.G;
    const int64_t n = P.ngp * S.ns;
    const int run = skip_solved ? 16 : 4;
    const int64_t waves = (n + run - 1) / run;
    const unsigned nb = (unsigned)((waves + 3) / 4);
#define LK_FIN(NJ)                                                                          \
  k_finalize<NJ><<<nb, 256, 0, st>>>(L, S, V, P, D, F.rtps, F.rtpp, F.mul, ana, F.amean,    \
                                     F.asprd, skip_solved, (uint32_t)n, run);               \
  break
    switch (((int)S.k + 15) / 16) {
      case 1: LK_FIN(1);
      case 2: LK_FIN(2);
      case 3: LK_FIN(3);
      case 4: LK_FIN(4);
      case 5: LK_FIN(5);
      case 6: LK_FIN(6);
      case 7: LK_FIN(7);
      default: LK_FIN(8);
    }
#undef LK_FIN
  }
}

}  // namespace lk
