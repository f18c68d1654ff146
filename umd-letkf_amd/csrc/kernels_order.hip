// kernels_order.hip -- list offsets and problem order of a chunk with few
// (gridpoint, group) pairs, one block each.
//
// A device-wide scan and a radix sort are 3 and 6 launches that each wait for
// the one before: with the copies of the totals, 55 us of a 360 us analysis
// (k = 10, 5 184 pairs) and 45 us of a 173 us replay (4 050).  Up to
// kSmallChunk (kSmallOrder) pairs a block of 1024 threads holds up to 16 each
// in registers; above, one block's share of memory bandwidth
// would cost more than the launches.
#include <hip/hip_runtime.h>

#include "letkf_internal.h"

namespace lk {

constexpr int kOrderThreads = 1024;
constexpr int kScanItems = kSmallChunk / kOrderThreads, kOrderItems = kSmallOrder / kOrderThreads;

// off = exclusive sums of the padded counts.  cap >= 0 (captured analysis):
// k_list_guard's check of every pair against the list capacity as well;
// tot (eager): the last pair's offset and count and the search counters go
// to page-locked memory (k_counters_to_host).
__global__ __launch_bounds__(kOrderThreads) void k_scan_small(int np, int64_t* cnt, int64_t* off,
                                                              uint8_t* solve, int64_t cap,
                                                              unsigned long long* ctr,
                                                              unsigned long long* h_ctr,
                                                              int64_t* tot) {
  __shared__ int64_t ws[kOrderThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int per = (np + kOrderThreads - 1) / kOrderThreads, p0 = tid * per;
  int64_t c[kScanItems], sum = 0;
#pragma unroll
  for (int e = 0; e < kScanItems; ++e) c[e] = e < per && p0 + e < np ? cnt[p0 + e] : 0;
#pragma unroll
  for (int e = 0; e < kScanItems; ++e) sum += PadCount()(c[e]);
  int64_t x = sum;                       // inclusive over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) ws[wv] = x;
  __syncthreads();
  int64_t at = x - sum;
  for (int w = 0; w < wv; ++w) at += ws[w];
#pragma unroll
  for (int e = 0; e < kScanItems; ++e) {
    const int p = p0 + e;
    if (e >= per || p >= np) continue;
    off[p] = at;
    if (tot && p == np - 1) {
      tot[0] = at;
      tot[1] = c[e];
    }
    at += PadCount()(c[e]);
    if (cap >= 0 && at + kListAlign > cap) {
      cnt[p] = 0;
      solve[p] = 0;
      atomicAdd(ctr + kCtrOverflow, 1ull);
    }
  }
  if (tot && tid < kCtrSlots * kCtrStride / kCtrStep) h_ctr[tid * kCtrStep] = ctr[tid * kCtrStep];
}

// perm: the problems by buckets of the kept count, largest first (bucket_desc);
// within a bucket roughly in gridpoint order, as the atomics come; no result
// depends on it
__global__ __launch_bounds__(kOrderThreads) void k_order_small(int np, int bbits,
                                                               const int64_t* __restrict__ cnt,
                                                               const uint8_t* __restrict__ solve,
                                                               int32_t* __restrict__ perm) {
  constexpr int NB = 128;                // 32 << bbits, bbits <= 2
  __shared__ int base[NB];
  const int tid = threadIdx.x;
  if (tid < NB) base[tid] = 0;
  __syncthreads();
  uint32_t b[kOrderItems];
#pragma unroll
  for (int e = 0; e < kOrderItems; ++e) {
    const int p = e * kOrderThreads + tid;
    b[e] = p < np ? bucket_desc(solve[p] ? cnt[p] : 0, bbits) : 0;
  }
#pragma unroll
  for (int e = 0; e < kOrderItems; ++e)
    if (e * kOrderThreads + tid < np) atomicAdd(&base[b[e]], 1);
  __syncthreads();
  if (tid < 64) {                        // exclusive sums of the bucket sizes
    const int n0 = base[2 * tid], n1 = base[2 * tid + 1];
    int x = n0 + n1;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (tid >= o) x += y;
    }
    base[2 * tid] = x - n0 - n1;
    base[2 * tid + 1] = x - n1;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kOrderItems; ++e) {
    const int p = e * kOrderThreads + tid;
    if (p < np) perm[atomicAdd(&base[b[e]], 1)] = p;
  }
}

void launch_scan_small(hipStream_t st, int64_t np, int64_t* cnt, int64_t* off, uint8_t* solve,
                       int64_t cap, unsigned long long* ctr, unsigned long long* h_ctr,
                       int64_t* tot) {
  k_scan_small<<<1, kOrderThreads, 0, st>>>((int)np, cnt, off, solve, cap, ctr, h_ctr, tot);
}

void launch_order_small(hipStream_t st, int64_t np, int bbits, const int64_t* cnt,
                        const uint8_t* solve, int32_t* perm) {
  k_order_small<<<1, kOrderThreads, 0, st>>>((int)np, bbits, cnt, solve, perm);
}

}  // namespace lk
