// kernels_ingest.hip -- the steps either side of the local analysis:
//
//  k_state_from_members  letkf_state_init (src/letkf_state.F90:326-334): from
//                        the members in file order (gridpoint fastest, then
//                        slab, then member) to state_ij(k, ns, ij) background
//                        perturbations, the mean SUM(.,1)/ens_size and the
//                        spread SQRT(DOT_PRODUCT(x', x')/(ens_size - 1)), in
//                        FP32 with the reference's order of operations
//  k_members_from_state  the analysis back to file order (the layout change of
//                        letkf_state_write_ens, :877-955) and the mean and
//                        spread (letkf_state_write_meansprd, :357-451)
//  k_obs_hx_split        letkf_obs_read (src/letkf_obs.F90:459-466):
//                        obs_hx_mean = SUM(obs_hx, 1)/ens_size and the
//                        perturbations obs_hx - obs_hx_mean, FP32
//  k_obs_compact         the QC compaction of :479-489 (qc > 0 dropped, order
//                        kept) as a gather through the selected indices
//  k_f64_to_f32          the FP32 view of the analysis (state_ij's REAL kind)
//  k_state_to_host, k_diag_to_host, k_counters_to_host
//                        results written into page-locked host memory
#include <hip/hip_runtime.h>

#include <algorithm>

#include "letkf_internal.h"

namespace lk {

#pragma clang fp contract(off)

// members[ij + nij * (s + ns * m)]: a block takes kTileGp gridpoints of a slab
// through LDS (rows of odd length), so that both orders are read and written
// in whole lines; one thread a gridpoint adds its members in the reference's
// order.  With a thread walking its own column in memory, 259 200 gridpoints
// of k = 50 took 168 us in and 141 us out, at a third of the copy rate.
constexpr int kTileGp = 64;
__global__ __launch_bounds__(256) void k_state_from_members(int64_t nij, int64_t ns, int k,
                                                            const float* __restrict__ members,
                                                            float* __restrict__ state,
                                                            float* __restrict__ mean,
                                                            float* __restrict__ sprd) {
  extern __shared__ float tile[];
  __shared__ float smu[kTileGp];
  const int ld = k | 1;
  const int64_t nt = (nij + kTileGp - 1) / kTileGp;
  const int64_t s = blockIdx.x / nt, i0 = (blockIdx.x - s * nt) * kTileGp;
  const int ng = (int)min((int64_t)kTileGp, nij - i0);
  const int64_t stride = nij * ns;
  const int g = threadIdx.x % kTileGp;
  if (g < ng) {
    const float* x = members + i0 + g + nij * s;
    for (int m = threadIdx.x / kTileGp; m < k; m += 256 / kTileGp) tile[g * ld + m] = x[m * stride];
  }
  __syncthreads();
  if ((int)threadIdx.x < ng) {
    const float* x = tile + g * ld;
    float sum = 0.0f;
    for (int m = 0; m < k; ++m) sum = sum + x[m];
    const float mu = sum / (float)k;
    float dot = 0.0f;
    for (int m = 0; m < k; ++m) {
      const float d = x[m] - mu;
      dot = dot + d * d;
    }
    smu[g] = mu;
    mean[s + ns * (i0 + g)] = mu;
    sprd[s + ns * (i0 + g)] = sqrtf(dot / (float)(k - 1));
  }
  __syncthreads();
  for (int e = threadIdx.x; e < ng * k; e += 256) {
    const int q = e / k, m = e % k;
    state[(int64_t)k * (s + ns * (i0 + q)) + m] = tile[q * ld + m] - smu[q];
  }
}

// analysis (FP64 on the device) to FP32 file order
__global__ __launch_bounds__(256) void k_members_from_state(int64_t nij, int64_t ns, int k,
                                                            const double* __restrict__ ana,
                                                            const double* __restrict__ amean,
                                                            const double* __restrict__ asprd,
                                                            float* __restrict__ members,
                                                            float* __restrict__ mean,
                                                            float* __restrict__ sprd) {
  extern __shared__ float tile[];
  const int ld = k | 1;
  const int64_t nt = (nij + kTileGp - 1) / kTileGp;
  const int64_t s = blockIdx.x / nt, i0 = (blockIdx.x - s * nt) * kTileGp;
  const int ng = (int)min((int64_t)kTileGp, nij - i0);
  const int64_t stride = nij * ns;
  const int g = threadIdx.x % kTileGp;
  if (members) {
    for (int e = threadIdx.x; e < ng * k; e += 256) {
      const int q = e / k, m = e % k;
      tile[q * ld + m] = (float)ana[(int64_t)k * (s + ns * (i0 + q)) + m];
    }
    __syncthreads();
    if (g < ng) {
      float* x = members + i0 + g + nij * s;
      for (int m = threadIdx.x / kTileGp; m < k; m += 256 / kTileGp) x[m * stride] = tile[g * ld + m];
    }
  }
  if ((int)threadIdx.x < ng) {
    if (mean) mean[i0 + g + nij * s] = (float)amean[s + ns * (i0 + g)];
    if (sprd) sprd[i0 + g + nij * s] = (float)asprd[s + ns * (i0 + g)];
  }
}

// hx (k, n) full values in, mean and perturbations out; flag = qc <= 0 (kept).
// A block stages the columns of kSplitObs observations in LDS (rows of odd
// length), whole lines in and out of memory; one thread an observation adds
// its members in the reference's order.  With a thread reading its own column
// from memory, 500 000 observations of k = 50 took 990 us.
constexpr int kSplitObs = 32;
__global__ __launch_bounds__(256) void k_obs_hx_split(int64_t n, int k,
                                                      const float* __restrict__ hx,
                                                      const int32_t* __restrict__ qc,
                                                      float* __restrict__ pert,
                                                      float* __restrict__ hmean,
                                                      uint8_t* __restrict__ keep) {
  extern __shared__ float tile[];
  __shared__ float smu[kSplitObs];
  const int ld = k | 1;
  const int64_t i0 = (int64_t)blockIdx.x * kSplitObs;
  const int no = (int)min((int64_t)kSplitObs, n - i0);
  const float* x = hx + (int64_t)k * i0;
  for (int e = threadIdx.x; e < no * k; e += 256) tile[e / k * ld + e % k] = x[e];
  __syncthreads();
  if ((int)threadIdx.x < no) {
    const float* t = tile + threadIdx.x * ld;
    float sum = 0.0f;
    for (int m = 0; m < k; ++m) sum = sum + t[m];
    const float mu = sum / (float)k;
    smu[threadIdx.x] = mu;
    hmean[i0 + threadIdx.x] = mu;
    keep[i0 + threadIdx.x] = qc[i0 + threadIdx.x] <= 0 ? 1 : 0;
  }
  __syncthreads();
  float* p = pert + (int64_t)k * i0;
  for (int e = threadIdx.x; e < no * k; e += 256) p[e] = tile[e / k * ld + e % k] - smu[e / k];
}

// gather the kept observations (sel: their indices in input order); the
// field pointers travel by value (their columns: launch_gather_cols)
__global__ void k_obs_compact(int64_t nsel, const int32_t* __restrict__ sel,
                              ObsFields in, ObsFields out) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nsel) return;
  const int64_t i = sel[j];
#pragma unroll
  for (int f = 0; f < ObsFields::kF; ++f) out.f[f][j] = in.f[f][i];
#pragma unroll
  for (int f = 0; f < ObsFields::kI; ++f) out.i[f][j] = in.i[f][i];
}

// FP64 -> FP32 (round to nearest), grid-stride over n values
__global__ void k_f64_to_f32(int64_t n, const double* __restrict__ in, float* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = (float)in[i];
}

// The analysis straight into the caller's page-locked arrays, in one launch:
// state, mean and spread converted to O (float rounds to nearest, double is a
// copy) and written over the bus by the lanes, four values each where the
// array starts on 16 bytes.  A staging buffer, a conversion and a copy for
// each array, each waited for, cost 100 us on a grid whose copies take 12;
// on large ones the conversion now runs in the copy's time.
struct ToHost {
  const double* src[3];
  void* dst[3];
  int64_t n[3];
};
template <typename O>
__global__ __launch_bounds__(256) void k_state_to_host(ToHost T) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  typedef O Ox __attribute__((ext_vector_type(16 / sizeof(O))));
  constexpr int W = 16 / sizeof(O);
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    const double* __restrict__ in = T.src[f];
    O* __restrict__ out = (O*)T.dst[f];
    const int64_t n = T.n[f];
    int64_t done = 0;
    if ((reinterpret_cast<uintptr_t>(out) & 15) == 0) {
      const int64_t nv = n / W;
      for (int64_t i = i0; i < nv; i += stride) {
        Ox v;
#pragma unroll
        for (int e = 0; e < W; ++e) v[e] = (O)in[W * i + e];
        __builtin_nontemporal_store(v, reinterpret_cast<Ox*>(out) + i);
      }
      done = nv * W;
    }
    for (int64_t i = done + i0; i < n; i += stride) out[i] = (O)in[i];
  }
}

void launch_state_to_host(hipStream_t st, bool f64, const double* const* src, void* const* dst,
                          const int64_t* n) {
  ToHost T;
  int64_t most = 0;
  for (int f = 0; f < 3; ++f) {
    T.src[f] = src[f];
    T.dst[f] = dst[f];
    T.n[f] = dst[f] ? n[f] : 0;
    most = std::max(most, T.n[f]);
  }
  if (most <= 0) return;
  const unsigned nb = (unsigned)std::min<int64_t>((most + 1023) / 1024, 1024);
  if (f64) k_state_to_host<double><<<nb, 256, 0, st>>>(T);
  else k_state_to_host<float><<<nb, 256, 0, st>>>(T);
}

// The diagnostics fields of an analysis as letkf_gpu_get_diag returns them,
// in page-locked memory: maxhz, obscount (nij), then per (group, gridpoint)
// kept count, weight sum (FP32) and hash
__global__ __launch_bounds__(256) void k_diag_to_host(int64_t nij, int64_t G, DiagDev D,
                                                      uint64_t* __restrict__ hash,
                                                      float* __restrict__ f) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nij * G) return;
  const int64_t g = e / nij, i = e - g * nij;
  if (g == 0) {
    f[i] = D.maxhz[i];
    f[nij + i] = (float)D.obscount[i];
  }
  hash[e] = D.lg_hash[i * G + g];
  f[2 * nij + e] = (float)D.lg_m[i * G + g];
  f[(2 + G) * nij + e] = (float)D.lg_obsloc[i * G + g];
}

void launch_diag_to_host(hipStream_t st, int64_t nij, int64_t G, const DiagDev& D,
                         uint64_t* hash, float* f) {
  if (nij * G <= 0) return;
  k_diag_to_host<<<(unsigned)((nij * G + 255) / 256), 256, 0, st>>>(nij, G, D, hash, f);
}

// the search counters (every kCtrStep-th word of a slot) and, where tot is
// given, the last pair's list offset and count, into page-locked memory
__global__ __launch_bounds__(256) void k_counters_to_host(const unsigned long long* ctr,
                                                          unsigned long long* h_ctr,
                                                          const int64_t* off, const int64_t* cnt,
                                                          int64_t* tot) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e < kCtrSlots * kCtrStride / kCtrStep) h_ctr[e * kCtrStep] = ctr[e * kCtrStep];
  if (tot && e == 0) {
    tot[0] = *off;
    tot[1] = *cnt;
  }
}

void launch_counters_to_host(hipStream_t st, const unsigned long long* ctr,
                             unsigned long long* h_ctr, const int64_t* off, const int64_t* cnt,
                             int64_t* tot) {
  k_counters_to_host<<<(kCtrSlots * kCtrStride / kCtrStep + 255) / 256, 256, 0, st>>>(
      ctr, h_ctr, off, cnt, tot);
}

void launch_f64_to_f32(hipStream_t st, int64_t n, const double* in, float* out) {
  if (n <= 0) return;
  const int64_t nb = std::min<int64_t>((n + 255) / 256, 8192);
  k_f64_to_f32<<<(unsigned)nb, 256, 0, st>>>(n, in, out);
}

void launch_state_from_members(hipStream_t st, int64_t nij, int64_t ns, int k,
                               const float* members, float* state, float* mean, float* sprd) {
  if (nij * ns <= 0) return;
  const int64_t nb = (nij + kTileGp - 1) / kTileGp * ns;
  k_state_from_members<<<(unsigned)nb, 256, sizeof(float) * kTileGp * (k | 1), st>>>(
      nij, ns, k, members, state, mean, sprd);
}

void launch_members_from_state(hipStream_t st, int64_t nij, int64_t ns, int k,
                               const double* ana, const double* amean, const double* asprd,
                               float* members, float* mean, float* sprd) {
  if (nij * ns <= 0) return;
  const int64_t nb = (nij + kTileGp - 1) / kTileGp * ns;
  k_members_from_state<<<(unsigned)nb, 256, sizeof(float) * kTileGp * (k | 1), st>>>(
      nij, ns, k, ana, amean, asprd, members, mean, sprd);
}

void launch_obs_hx_split(hipStream_t st, int64_t n, int k, const float* hx, const int32_t* qc,
                         float* pert, float* hmean, uint8_t* keep) {
  if (n <= 0) return;
  k_obs_hx_split<<<(unsigned)((n + kSplitObs - 1) / kSplitObs), 256,
                   sizeof(float) * kSplitObs * (k | 1), st>>>(n, k, hx, qc, pert, hmean, keep);
}

void launch_obs_compact(hipStream_t st, int64_t nsel, int k, const int32_t* sel,
                        const ObsFields& in, const ObsFields& out) {
  if (nsel <= 0) return;
  k_obs_compact<<<(unsigned)((nsel + 255) / 256), 256, 0, st>>>(nsel, sel, in, out);
  launch_gather_cols(st, nsel, k, sel, in.hx, out.hx);
}

}  // namespace lk
