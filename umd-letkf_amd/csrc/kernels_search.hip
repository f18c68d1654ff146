// kernels_search.hip -- local-observation search and localization.
//
// Replaces, per gridpoint, the reference's
//   maxhz / search radius ........ src/letkf_solver.F90:210-212
//   kd_search_radius ............. src/letkf_obs.F90:560-573
//   groups() ..................... letkf_loc_novrt.F90:133-147,
//                                  letkf_loc_ocean.F90:331-427
//   localize() + keep r > 1e-4 ... src/letkf_solver.F90:244-268,
//                                  letkf_loc_novrt.F90:170-183,
//                                  letkf_loc_ocean.F90:451-506
//
// One 64-lane wavefront owns one gridpoint.  The gridpoint's search cap is
// covered by whole lat/lon cells (a conservative superset computed with
// margins); lanes stride over the contiguous obs ranges of those cells and
// apply the exact test (squared chord <= threshold) and the localizer in
// the deterministic arithmetic of det_math.h.  Kept observations are counted
// per localization group with ballots.  The same kernel runs twice: the
// count pass sizes the lists, the fill pass writes each (gridpoint,
// group)'s kept (obs index, weight) list in scan order.  With several
// groups the count pass localizes (exact counts, diagnostics); with one it
// only sums the cover's cell sizes, and the fill pass writes the
// diagnostics.
#include <hip/hip_runtime.h>

#include "det_math.h"
#include "eigen_common.h"
#include "letkf_internal.h"

namespace lk {

constexpr double kRad2Deg = 57.295779513082320876;

__device__ __forceinline__ double wave_sum_f64(double v) { return wave_sum_dpp(v); }
template <int CTRL, int ROWMASK>
__device__ __forceinline__ uint64_t dpp_u64(uint64_t v) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROWMASK, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWMASK, 0xf, false);
  return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}
__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
  v += dpp_u64<0x111, 0xf>(v);
  v += dpp_u64<0x112, 0xf>(v);
  v += dpp_u64<0x114, 0xf>(v);
  v += dpp_u64<0x118, 0xf>(v);
  v += dpp_u64<0x142, 0xa>(v);
  v += dpp_u64<0x143, 0xc>(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), 63);
  return ((uint64_t)hi << 32) | lo;
}
// exclusive prefix sum over the wave's lanes, and the total
__device__ __forceinline__ int wave_excl_scan(int v, int lane, int* total) {
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  *total = __shfl(x, 63, 64);
  return x - v;
}
__device__ __forceinline__ int lane_rank(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// vertical weight of one observation at level g (FP32 result)
__device__ __forceinline__ float vertical_weight(float vt_scale, float zdim, float depth) {
#pragma clang fp contract(off)
  const double dz = (double)zdim - (double)depth;
  const double sc = (double)vt_scale;
  return (float)dm::exp_neg(-(dz * dz) / (2.0 * sc * sc));
}

__device__ __forceinline__ bool group_has_slabs(int cls, const LocDev& L, int g, int mld) {
  if (cls == LETKF_LOC_OCEAN && L.vtloc_surf == 1) return g == 0 || L.max_var_lev > mld;
  if (cls == LETKF_LOC_VGAUSS) return g < L.max_var_lev;
  return true;
}

// dm::interp on a table held in the kernel arguments, with constant indices
// only (a table read at a computed index would make the compiler copy the
// whole argument block to private memory); the same arithmetic
__device__ __forceinline__ float interp_arg(int n, const float (&lat)[kTab],
                                            const float (&dist)[kTab], float x) {
#pragma clang fp contract(off)
  const float a = fabsf(x);
  int i = n - 1;
#pragma unroll
  for (int j = kTab - 1; j >= 0; --j)
    if (j < n - 1 && !(a > lat[j])) i = j;
  if (i == 0) return dist[0];
  float l1 = 0.0f, d1 = 0.0f, l0 = 0.0f, d0 = 0.0f;
#pragma unroll
  for (int j = 0; j < kTab; ++j) {
    if (j == i) { l1 = lat[j]; d1 = dist[j]; }
    if (j == i - 1) { l0 = lat[j]; d0 = dist[j]; }
  }
  const float d = (a - l0) / (l1 - l0);
  return d * d1 + (1.0f - d) * d0;
}

// Search radius of a gridpoint (src/letkf_solver.F90:210-212) and the
// localization distances it comes from.
struct Radii {
  float Lh, Lp, Ls, maxhz, rs;
};

__device__ __forceinline__ Radii search_radii(int cls, const LocDev& L, float lat_ij) {
  Radii R{0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  if (cls == LETKF_LOC_OCEAN) {
    R.Lp = interp_arg(L.n_prof, L.prof_lat, L.prof_dist, lat_ij);
    R.Ls = interp_arg(L.n_sat, L.sat_lat, L.sat_dist, lat_ij);
    R.maxhz = R.Lp > R.Ls ? R.Lp : R.Ls;
  } else {
    R.Lh = interp_arg(L.n_hz, L.hz_lat, L.hz_dist, lat_ij);
    R.maxhz = R.Lh;
  }
  {
#pragma clang fp contract(off)
    R.rs = R.maxhz * dm::kSTDEV2MAX;                  // src/letkf_solver.F90:211
  }
  return R;
}

// Conservative cell cover of a spherical cap: bands b0..b1 and, in each
// band, the longitude cells the cap can reach within that band.  The count
// pass and the fill pass use these same functions without contraction, so
// both compute the same cells and the list space the count pass sizes holds
// every candidate the fill pass scans.
struct CapCover {
  double lat0, lon0, thd, hav_cap, cos_lat0;
  int b0, b1;
  bool all_lon;   // the cap reaches a pole: whole bands
};

// cosine of a latitude in degrees, by det_math.h's polynomials (the
// library's sin, cos and asin carry range reductions that no argument here
// needs; the cover has margins far above the rounding)
__device__ __forceinline__ double cos_lat(double deg) {
  const double x = fabs(deg) / kRad2Deg;
  return x <= dm::kPIO4 ? dm::cos_core(x) : dm::sin_core(dm::kPIO2 - x);
}

__device__ __forceinline__ CapCover cap_cover(float rs, float lat, float lon) {
#pragma clang fp contract(off)
  CapCover cv;
  const double theta = (double)rs / dm::kRE * (1.0 + 1e-6) + 1e-9;
  cv.lat0 = (double)lat;
  cv.lon0 = (double)lon;
  cv.lon0 = cv.lon0 - 360.0 * floor(cv.lon0 / 360.0);
  cv.b0 = 0;
  cv.b1 = kBands - 1;
  cv.all_lon = true;
  cv.thd = 180.0;
  if (theta < 3.14159) {
    cv.thd = theta * kRad2Deg;
    int b0 = (int)floor(cv.lat0 - cv.thd + 90.0);
    int b1 = (int)floor(cv.lat0 + cv.thd + 90.0);
    cv.b0 = b0 < 0 ? 0 : (b0 >= kBands ? kBands - 1 : b0);
    cv.b1 = b1 < 0 ? 0 : (b1 >= kBands ? kBands - 1 : b1);
    cv.all_lon = !(cv.lat0 + cv.thd < 90.0 && cv.lat0 - cv.thd > -90.0);
  }
  const double sh = dm::sin_rad(fmin(0.5 * theta, 1.5));   // not used past a pole
  cv.hav_cap = sh * sh;
  cv.cos_lat0 = cos_lat(cv.lat0);
  return cv;
}

// longitude half-width (degrees) that bounds the cap within band b, from
//   hav(dlon) = (hav(cap) - hav(dlat)) / (cos lat0 cos lat),
// with dlat at its smallest over the band and |lat| at its largest over the
// band's part of the cap's latitude range; < 0: the band misses the cap.
// Bands past the 64th of the cover (caps wider than 32 degrees) take whole
// longitude circles.
__device__ __forceinline__ double cover_halfwidth(const CapCover& cv, int b) {
#pragma clang fp contract(off)
  if (cv.all_lon || b - cv.b0 >= 64) return 180.0;
  const double la = (double)b - 90.0, lb = la + 1.0;
  const double dmin = cv.lat0 < la ? la - cv.lat0 : (cv.lat0 > lb ? cv.lat0 - lb : 0.0);
  const double sd = dm::sin_rad(0.5 * dmin / kRad2Deg);
  const double num = cv.hav_cap - sd * sd;
  if (num <= 0.0) return -1.0;
  const double lo = fmax(la, cv.lat0 - cv.thd), hi = fmin(lb, cv.lat0 + cv.thd);
  const double amax = lo <= hi ? fmax(fabs(lo), fabs(hi)) : fmax(fabs(la), fabs(lb));
  const double q = num / (cv.cos_lat0 * cos_lat(amax));
  if (!(q < 1.0)) return 180.0;
  return 2.0 * dm::asin01(sqrt(q)) * kRad2Deg * (1.0 + 1e-9) + 1e-6;
}

// the one or two longitude cell ranges [rc0, rc1] of half-width dl (< 180)
__device__ __forceinline__ int cover_ranges(const CapCover& cv, double dl, int rc0[2],
                                            int rc1[2]) {
#pragma clang fp contract(off)
  rc0[0] = 0; rc0[1] = 0;
  rc1[0] = kLonCells - 1; rc1[1] = kLonCells - 1;
  if (!(dl < 180.0)) return 1;
  const int c0 = (int)floor(cv.lon0 - dl), c1 = (int)floor(cv.lon0 + dl);
  if (c0 < 0) { rc0[0] = c0 + kLonCells; rc1[0] = kLonCells - 1; rc0[1] = 0; rc1[1] = c1; return 2; }
  if (c1 >= kLonCells) { rc0[0] = c0; rc1[0] = kLonCells - 1; rc0[1] = 0; rc1[1] = c1 - kLonCells; return 2; }
  rc0[0] = c0;
  rc1[0] = c1;
  return 1;
}

// Passes (one wave per gridpoint):
//   kCountExact  kept counts and diagnostics per group (weights evaluated)
//   kFill        lists written at the offsets of the exact counts
//   kFillDiag    one group: lists written at the offsets of the bounds that
//                k_count_cover (below) sizes, then the kept count, the solve
//                flag, the search-set size and the other diagnostics
constexpr int kCountExact = 0, kFill = 1, kFillDiag = 3;
constexpr int kQueue = 128;   // per-wave candidate ring (two batches)
constexpr int kSeg = 256;     // several groups: localized candidates held back

// orders this wave's LDS stores and loads on either side (the queue is
// private to one wave; the block's waves retire independently, so no
// block barrier)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// sqrt(w / err) of the mixed products' lists, by the hardware reciprocal and
// square root (1 ulp each; the products round far more)
__device__ __forceinline__ float list_weight(float w, float err) {
  return __builtin_amdgcn_sqrtf(w * __builtin_amdgcn_rcpf(err));
}

// the one-group fill pass (the common case) keeps one group in LDS, which
// leaves five waves per SIMD to hide the candidates' load latency
template <int PASS, int CLS>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(PASS == 3 ? 5 : 1, 8))) void k_search(LocDev L, ObsDev O, StateDev S,
                                                VarsDev V, ChunkDev C, DiagDev D) {
  constexpr bool FILL = PASS == kFill || PASS == kFillDiag;
  constexpr bool STATS = PASS == kCountExact || PASS == kFillDiag;   // sums, hash
  constexpr int NG = PASS == kFillDiag ? 1 : kMaxGroups;   // groups held in LDS
  __shared__ int64_t s_cnt[4][NG];
  __shared__ double s_sum[4][NG];
  __shared__ uint64_t s_hash[4][NG];
  __shared__ int64_t s_lim[4][NG];               // fill: end of each list's space
  __shared__ int32_t s_qs[4][kQueue];             // queued candidates: obs index,
  __shared__ double s_qc[4][kQueue];              //   squared chord,
  __shared__ float s_qe[4][kQueue];               //   error variance
  __shared__ uint64_t s_qh[4][STATS ? kQueue : 1];   //   and index hash
  // several groups: horizontally localized candidates (observation, surface
  // flag in bit 31; weight; error variance or hash), in scan order
  constexpr bool SEG = PASS != kFillDiag;
  __shared__ int32_t s_gs[4][SEG ? kSeg : 1];
  __shared__ float s_gw[4][SEG ? kSeg : 1];
  __shared__ float s_ge[4][SEG && FILL ? kSeg : 1];
  __shared__ uint64_t s_gh[4][SEG && !FILL ? kSeg : 1];
  __shared__ int32_t s_rsb[4][129];               // cover ranges: first obs
  __shared__ int32_t s_roff[4][130];              //   and offset in the candidate stream
  const int wid = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + wid;
  if (t >= C.ngp) return;
  const int64_t ij = C.i0 + t;
  const int G = C.G;

  if (lane == 0) {
    for (int g = 0; g < G; ++g) {
      s_cnt[wid][g] = FILL ? C.off[t * G + g] : 0;
      s_lim[wid][g] = FILL ? C.off[t * G + g] + C.cnt[t * G + g] : 0;
      s_sum[wid][g] = 0.0;
      s_hash[wid][g] = 0;
    }
  }
  if (S.mask[ij]) {                                   // src/letkf_solver.F90:207
    if (PASS == kCountExact) {
      if (lane != 0) return;
      for (int g = 0; g < G; ++g) {
        C.cnt[t * G + g] = 0;
        C.solve[t * G + g] = 0;
        D.lg_m[ij * G + g] = 0;
        D.lg_obsloc[ij * G + g] = 0.0;
        D.lg_hash[ij * G + g] = 0;
      }
      D.obscount[ij] = 0;
      D.maxhz[ij] = 0.0f;
      D.mld[ij] = 0;
    }
    return;
  }

  const float lat_ij = S.lat[ij];
  const Radii R = search_radii(CLS, L, lat_ij);
  const float tloc_prof = L.tloc_prof, tloc_sat = L.tloc_sat, vt_scale = L.vt_scale;
  const float maxhz = R.maxhz, rs = R.rs;
  const double thr2 = dm::thr2(rs);
  // length scale of the weights (LOC_OCEAN: profile, and that of surface obs)
  const float L0 = CLS == LETKF_LOC_OCEAN ? R.Lp : R.Lh;
  const dm::GcScale gs0 = dm::gc_scale(L0);
  const dm::GcScale gs1 = CLS == LETKF_LOC_OCEAN ? dm::gc_scale(R.Ls) : gs0;
  const bool near_cap = 0.25 * thr2 <= dm::kFastHalf2;   // wave-uniform

  int mld = 0;                                        // calc_mldlvl_bkgt
  if (CLS == LETKF_LOC_OCEAN && L.vtloc_surf == 1) {
    const float* mean = S.mean + S.ns * ij;
    const float t0 = mean[L.bkg_t_var_idx];
    mld = L.bkg_t_var_len;
    for (int i = 1; i <= L.bkg_t_var_len - 1; ++i) {
      const float t1 = mean[L.bkg_t_var_idx + i];
      if (fabsf(t0 - t1) > L.bkg_t_delta) { mld = i; break; }
    }
  }

  const double gx = S.gx[ij], gy = S.gy[ij], gz = S.gz[ij];

  const CapCover cv = cap_cover(rs, lat_ij, S.lon[ij]);
  const int b0 = cv.b0, b1 = cv.b1;

  int64_t nin = 0, ncand = 0;
  double lsum = 0.0;          // kFillDiag: this lane's weights and hashes
  uint64_t lhash = 0;

  // Candidates inside the cap go through a per-wave queue in LDS (a ring of
  // 128 entries, in scan order) and are localized 64 at a time, so that the
  // distance, weight, hash and list work runs on full waves; lists are
  // written in the same scan order as without the queue.
  int qh = 0, qn = 0;          // ring head and length (wave-uniform)
  // one group: the list cursor and end stay in (wave-uniform) registers
  int64_t fd_cur = 0, fd_lim = 0;
  if (PASS == kFillDiag) {
    fd_cur = C.off[t];
    fd_lim = fd_cur + C.cnt[t];
  }
  int sn = 0;                  // several groups: candidates held back (wave-uniform)
  // Several groups: the candidates held back go through the groups 64 at a
  // time, with one reduction of the sums for each group and up to kSeg of
  // them (a reduction costs as much as 50 weights).  The count pass of 50
  // levels on 16 200 gridpoints: 3.6 ms with a reduction for every 64
  // candidates and the vertical weights evaluated each time, 1.7 ms now.
  auto flush = [&]() __attribute__((always_inline)) {
    wave_lds_fence();
    for (int g = 0; g < G; ++g) {
      const float depth = CLS == LETKF_LOC_VGAUSS ? V.lev_depth[g] : 0.0f;
      const float* vt = CLS == LETKF_LOC_VGAUSS && O.vt ? O.vt + g * O.n : nullptr;
      int64_t cur = 0, lim = 0;
      if (FILL) { cur = s_cnt[wid][g]; lim = s_lim[wid][g]; }
      int64_t kept = 0;
      double sum = 0.0;
      uint64_t hash = 0;
      for (int e0 = 0; e0 < sn; e0 += 64) {
        const int e = e0 + lane;
        const bool in = e < sn;
        const int32_t sv = in ? s_gs[wid][e] : 0;
        float w = in ? s_gw[wid][e] : 0.0f;
        const int32_t o = sv & 0x7fffffff;
        if (CLS == LETKF_LOC_VGAUSS) {
          // the same product as hz * (float)v of the weight function
          const float v = vt ? vt[o] : vertical_weight(vt_scale, O.zdim[o], depth);
          w = w * v;
        }
        if (CLS == LETKF_LOC_OCEAN && g == 1 && sv < 0) w = 0.0f;   // surface obs: SURF only
        const bool keep = in && (w > 1.0e-4f);   // src/letkf_solver.F90:251
        const uint64_t kmask = __ballot(keep);
        if (kmask == 0) continue;
        if (STATS) {
          sum += keep ? (double)w : 0.0;
          hash += keep ? s_gh[wid][in ? e : 0] : 0ull;
        }
        if (FILL && keep) {
          // writes never pass the end of this pair's list space
          const int64_t pos = cur + kept + lane_rank(kmask);
          if (pos < lim) {
            C.list_idx[pos] = C.list_mode ? (int32_t)((int64_t)o * O.kp * 4) : o;
            C.list_w[pos] = C.list_mode ? list_weight(w, s_ge[wid][e]) : w;
          }
        }
        kept += __popcll(kmask);
      }
      if (kept == 0) continue;
      if (STATS) {
        sum = wave_sum_f64(sum);
        hash = wave_sum_u64(hash);
      }
      if (lane == 0) {
        s_cnt[wid][g] += kept;
        if (STATS) {
          s_sum[wid][g] += sum;
          s_hash[wid][g] += hash;
        }
      }
    }
    sn = 0;
    wave_lds_fence();
  };
  auto localize = [&](int cnt) __attribute__((always_inline)) {
    wave_lds_fence();
    const bool inside = lane < cnt;
    const int e = (qh + lane) & (kQueue - 1);
    const int32_t s = inside ? s_qs[wid][e] : 0;
    const double c2 = inside ? s_qc[wid][e] : 1e-4;
    const float oerr = inside ? s_qe[wid][e] : 1.0f;
    const uint64_t mix = STATS && inside ? s_qh[wid][STATS ? e : 0] : 0ull;
    bool surf = false;
    float tw = 1.0f;
    if (CLS == LETKF_LOC_OCEAN) {
      surf = inside && O.surf[s] != 0;
      if (surf && tloc_sat > 0.0f) tw = O.tw_sat[s];
      if (!surf && tloc_prof > 0.0f) tw = O.tw_prof[s];
    }
    wave_lds_fence();
    // the short forms, and the full ones where a lane is not sure of its float
    bool sure = false;
    float d = dm::dist_fast(c2, &sure);
    sure = sure && near_cap;
    if (__ballot(inside && !sure) != 0ull) {
      if (!sure) d = dm::dist(c2);
    }
    dm::GcScale gs = gs0;
    if (CLS == LETKF_LOC_OCEAN && surf) gs = gs1;
    float hz = dm::gc_fast(d, gs, &sure);
    if (__ballot(inside && !sure) != 0ull) {
      if (!sure) hz = dm::gc(d, CLS == LETKF_LOC_OCEAN && surf ? R.Ls : L0);
    }
    if (CLS == LETKF_LOC_OCEAN && (surf ? tloc_sat : tloc_prof) > 0.0f) hz = hz * tw;
    const bool keep = inside && (hz > 1.0e-4f);   // src/letkf_solver.F90:251
    const uint64_t kmask = __ballot(keep);
    if (PASS == kFillDiag) {
      // one group: per-lane partial sums, reduced once per gridpoint
      lsum += keep ? (double)hz : 0.0;
      lhash += keep ? mix : 0ull;
      if (keep) {
        // writes never pass the end of this pair's list space
        const int64_t pos = fd_cur + lane_rank(kmask);
        if (pos < fd_lim) {
          C.list_idx[pos] = C.list_mode ? (int32_t)((int64_t)s * O.kp * 4) : s;
          C.list_w[pos] = C.list_mode ? list_weight(hz, oerr) : hz;
        }
      }
      fd_cur += __popcll(kmask);
    } else if (kmask != 0) {
      // a group's weight is at most hz: what hz drops, every group drops
      if (sn + 64 > kSeg) flush();
      if (keep) {
        const int at = sn + lane_rank(kmask);
        s_gs[wid][at] = s | (surf ? (int32_t)0x80000000 : 0);
        s_gw[wid][at] = hz;
        if (FILL) s_ge[wid][FILL ? at : 0] = oerr;
        else s_gh[wid][FILL ? 0 : at] = mix;
      }
      sn += __popcll(kmask);
    }
    qh = (qh + cnt) & (kQueue - 1);
    qn -= cnt;
  };

  // The cover's cells: lane i finds the one or two longitude ranges of band
  // b0 + i and their obs ranges; bands past the 64th of the cover take whole
  // longitude circles, which follow one another in the cell order and make
  // one more range.  The ranges, in band order, make one stream of
  // candidates, scanned 64 at a time in the same order as band by band.  The
  // positions (and the fields the localization needs) of a batch are loaded
  // two batches ahead.
  const bool need_err = FILL && C.list_mode;
  struct Cand {
    double2 xy, zh;     // position, and the index hash
    float e;
    int32_t s;          // < 0: past the stream
  };
  {
    const int b = b0 + lane;
    int nr = 0, sb0 = 0, len0 = 0, sb1 = 0, len1 = 0;
    if (b <= b1) {
      const double dl = cover_halfwidth(cv, b);
      if (dl >= 0.0) {
        int rc0[2], rc1[2];
        nr = cover_ranges(cv, dl, rc0, rc1);
        const int32_t* cs = O.cell_start + b * kLonCells;
        sb0 = cs[rc0[0]];
        len0 = cs[rc1[0] + 1] - sb0;
        if (nr == 2) {
          sb1 = cs[rc0[1]];
          len1 = cs[rc1[1] + 1] - sb1;
        }
      }
    }
    int nrt = 0, T = 0;
    const int slot = wave_excl_scan(nr, lane, &nrt);
    const int off = wave_excl_scan(len0 + len1, lane, &T);
    if (nr >= 1) {
      s_rsb[wid][slot] = sb0;
      s_roff[wid][slot] = off;
    }
    if (nr == 2) {
      s_rsb[wid][slot + 1] = sb1;
      s_roff[wid][slot + 1] = off + len0;
    }
    if (b1 - b0 >= 64) {
      const int st0 = O.cell_start[(b0 + 64) * kLonCells];
      const int st1 = O.cell_start[(b1 + 1) * kLonCells];
      if (lane == 0) {
        s_rsb[wid][nrt] = st0;
        s_roff[wid][nrt] = T;
      }
      nrt += 1;
      T += st1 - st0;
    }
    if (lane == 0) s_roff[wid][nrt] = T;
    wave_lds_fence();
    if (PASS != kFill) ncand += T;
    int rl = 0;                       // range of this lane's next load
    // the loads are issued by every lane (past the stream: observation 0),
    // so that the wait for a batch counts the loads issued after it
    auto fetch = [&](Cand& c, int q) __attribute__((always_inline)) {
      const int p = q + lane;
      int so = 0;
      if (p < T) {
        while (p >= s_roff[wid][rl + 1]) ++rl;
        so = s_rsb[wid][rl] + (p - s_roff[wid][rl]);
      }
      c.s = p < T ? so : -1;
      c.xy = O.pos[2 * (int64_t)so];
      c.zh = O.pos[2 * (int64_t)so + 1];
      if (FILL) c.e = O.err[so];
    };
    auto scan = [&](const Cand& c) __attribute__((always_inline)) {
      double c2 = 9.0;
      if (c.s >= 0) c2 = dm::chord2(c.xy.x, c.xy.y, c.zh.x, gx, gy, gz);
      const bool inside = c2 <= thr2;
      const uint64_t imask = __ballot(inside);
      if (imask == 0) return;
      nin += __popcll(imask);
      // qn < 64 here, so the ring (128) has room for the whole batch
      if (inside) {
        const int e = (qh + qn + lane_rank(imask)) & (kQueue - 1);
        s_qs[wid][e] = c.s;
        s_qc[wid][e] = c2;
        s_qe[wid][e] = need_err ? c.e : 1.0f;
        if (STATS) s_qh[wid][STATS ? e : 0] = (uint64_t)__double_as_longlong(c.zh.y);
      }
      qn += __popcll(imask);
      if (qn >= 64) localize(64);
    };
    // three batches in registers, each in the same ones throughout (the
    // loop is unrolled three times, so no batch is moved while its loads
    // are in flight): the one scanned and the two loading
    Cand ca, cb, cc;
    if (T > 0) {
      fetch(ca, 0);
      fetch(cb, 64);
    }
    for (int q = 0; q < T; q += 192) {
      fetch(cc, q + 128);
      scan(ca);
      if (q + 64 >= T) break;
      fetch(ca, q + 192);
      scan(cb);
      if (q + 128 >= T) break;
      fetch(cb, q + 256);
      scan(cc);
    }
    wave_lds_fence();
  }
  if (qn > 0) localize(qn);
  if (PASS != kFillDiag && sn > 0) flush();

  if (PASS == kFillDiag) {
    const double sr = wave_sum_f64(lsum);
    const uint64_t hs = wave_sum_u64(lhash);
    if (lane == 0) {
      s_sum[wid][0] = sr;
      s_hash[wid][0] = hs;
      // the kept count never exceeds the list space the count pass sized
      // (the cover bound); a pair whose space was withdrawn (list capacity
      // guard) ends with no list
      s_cnt[wid][0] = fd_cur < fd_lim ? fd_cur : fd_lim;
    }
  }
  if (FILL && C.list_mode) {
    // zero the alignment padding after each list: the mixed products read
    // whole 8-entry groups
    for (int g = 0; g < G; ++g) {
      int64_t end = 0;
      if (lane == 0) {
        end = s_cnt[wid][g];
        const int64_t lim = PASS == kFillDiag ? fd_lim : s_lim[wid][g];
        if (end > lim) end = lim;      // only past the space of a guarded pair
      }
      end = __shfl(end, 0, 64);
      const int64_t pad_end = C.off[t * G + g] + PadCount()(end - C.off[t * G + g]);
      if (end + lane < pad_end) {
        C.list_idx[end + lane] = 0;
        C.list_w[end + lane] = 0.0f;
      }
    }
  }
  if (lane != 0 || PASS == kFill) return;
  unsigned long long* c = D.ctr + (blockIdx.x & (kCtrSlots - 1)) * kCtrStride;
  if (PASS == kCountExact || PASS == kFillDiag) {
    unsigned long long nsolve = 0, npair = 0;
    for (int g = 0; g < G; ++g) {
      const int64_t m = PASS == kFillDiag ? s_cnt[wid][g] - C.off[t * G + g] : s_cnt[wid][g];
      const bool sv = m > 0 && group_has_slabs(CLS, L, g, mld);
      nsolve += sv ? 1 : 0;
      npair += sv ? (unsigned long long)m : 0ull;
      C.cnt[t * G + g] = m;
      C.solve[t * G + g] = sv ? 1 : 0;
      D.lg_m[ij * G + g] = (int32_t)m;
      D.lg_obsloc[ij * G + g] = s_sum[wid][g];
      D.lg_hash[ij * G + g] = s_hash[wid][g];
    }
    atomicAdd(c + kCtrSolves, nsolve);
    atomicAdd(c + kCtrPairs, npair);
  }
  if (PASS == kCountExact || PASS == kFillDiag) {
    D.obscount[ij] = (int32_t)nin;
    D.maxhz[ij] = maxhz;
    D.mld[ij] = mld;
    atomicMax(c + kCtrMax, (unsigned long long)nin);
    atomicAdd(c + kCtrCand, (unsigned long long)ncand);
  }
}

// One-group count pass, eight lanes per gridpoint (a band each; on a small
// grid one lane walking the bands was a 45 us chain): the number of
// observations in the cells of the cap's cover, an upper bound of the kept
// count that sizes the list (the fill pass scans the same cells).  Masked
// gridpoints get zero counts and diagnostics.
__global__ __launch_bounds__(256) void k_count_cover(LocDev L, ObsDev O, StateDev S,
                                                     ChunkDev C, DiagDev D) {
  const int64_t t = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 3;
  const int l8 = threadIdx.x & 7;
  if (t >= C.ngp) return;
  const int64_t ij = C.i0 + t;
  if (S.mask[ij]) {                                   // src/letkf_solver.F90:207
    if (l8 != 0) return;
    C.cnt[t] = 0;
    C.solve[t] = 0;
    D.lg_m[ij] = 0;
    D.lg_obsloc[ij] = 0.0;
    D.lg_hash[ij] = 0;
    D.obscount[ij] = 0;
    D.maxhz[ij] = 0.0f;
    D.mld[ij] = 0;
    return;
  }
  const float lat_ij = S.lat[ij];
  const CapCover cv = cap_cover(search_radii(L.cls, L, lat_ij).rs, lat_ij, S.lon[ij]);
  int ncand = 0;
  for (int b = cv.b0 + l8; b <= cv.b1; b += 8) {
    const double dl = cover_halfwidth(cv, b);
    if (dl < 0.0) continue;
    int rc0[2], rc1[2];
    const int nr = cover_ranges(cv, dl, rc0, rc1);
    for (int r = 0; r < nr; ++r)
      ncand += O.cell_start[b * kLonCells + rc1[r] + 1] - O.cell_start[b * kLonCells + rc0[r]];
  }
  ncand += __shfl_xor(ncand, 1, 8);
  ncand += __shfl_xor(ncand, 2, 8);
  ncand += __shfl_xor(ncand, 4, 8);
  if (l8 == 0) C.cnt[t] = ncand;
}

// The graph-captured analysis.  Its counters are cleared by a kernel (a
// captured graph holds no memset nodes), and the list space is checked on
// the device instead of by the host: a (gridpoint, group) pair whose padded
// list (plus the alignment slack of the vector loads) would end past the
// list capacity gets no list space and no solve, and the overflow is
// counted for the host, which reads the counters after the replay.
__global__ void k_clear_u64(int64_t n, unsigned long long* p) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

__global__ void k_list_guard(int64_t np, int64_t* cnt, const int64_t* off, uint8_t* solve,
                             int64_t cap, unsigned long long* ctr) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  if (off[p] + PadCount()(cnt[p]) + kListAlign > cap) {
    cnt[p] = 0;
    solve[p] = 0;
    atomicAdd(ctr + kCtrOverflow, 1ull);
  }
}

void launch_clear_u64(hipStream_t st, int64_t n, unsigned long long* p) {
  if (n <= 0) return;
  k_clear_u64<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(n, p);
}

void launch_list_guard(hipStream_t st, int64_t np, int64_t* cnt, const int64_t* off,
                       uint8_t* solve, int64_t cap, unsigned long long* ctr) {
  if (np <= 0) return;
  k_list_guard<<<(unsigned)((np + 255) / 256), 256, 0, st>>>(np, cnt, off, solve, cap, ctr);
}

// the search kernel for localizer class CLS (its branches folded away)
template <int CLS>
static void launch_search_cls(hipStream_t st, int pass, unsigned nb, const LocDev& L,
                              const ObsDev& O, const StateDev& S, const VarsDev& V,
                              const ChunkDev& C, const DiagDev& D) {
  if (pass == kFillDiag) k_search<kFillDiag, CLS><<<nb, 256, 0, st>>>(L, O, S, V, C, D);
  else if (pass == kFill) k_search<kFill, CLS><<<nb, 256, 0, st>>>(L, O, S, V, C, D);
  else k_search<kCountExact, CLS><<<nb, 256, 0, st>>>(L, O, S, V, C, D);
}

void launch_search(hipStream_t st, bool fill, const LocDev& L, const ObsDev& O,
                   const StateDev& S, const VarsDev& V, const ChunkDev& C,
                   const DiagDev& D) {
  if (C.ngp <= 0) return;
  const unsigned nb = (unsigned)((C.ngp + 3) / 4);
  // one group: size the lists by the search set (chord test only) and count
  // the kept observations while writing them
  if (C.G == 1 && !fill) {
    k_count_cover<<<(unsigned)((C.ngp + 31) / 32), 256, 0, st>>>(L, O, S, C, D);
    return;
  }
  const int pass = C.G == 1 ? kFillDiag : (fill ? kFill : kCountExact);
  switch (L.cls) {
    case LETKF_LOC_OCEAN: launch_search_cls<LETKF_LOC_OCEAN>(st, pass, nb, L, O, S, V, C, D); break;
    case LETKF_LOC_VGAUSS: launch_search_cls<LETKF_LOC_VGAUSS>(st, pass, nb, L, O, S, V, C, D); break;
    default: launch_search_cls<LETKF_LOC_NOVRT>(st, pass, nb, L, O, S, V, C, D); break;
  }
}

}  // namespace lk
