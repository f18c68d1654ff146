// tridiag_pair.hip -- choice of the DPP tridiagonalization by row length (a
// multiple of 8 >= k, or 50 for k = 49 and 50; two problems per wave up to
// 50, one above: longer rows leave too few registers for two of them).
#include "letkf_internal.h"

namespace lk {

#define LK_DECL(KQ)                                                                     \
  int launch_tridiag_pair_##KQ(hipStream_t, int64_t, const int32_t*, int, int, int,     \
                               const LocDev&, const StateDev&, const VarsDev&,          \
                               const ChunkDev&, const DiagDev&, double*, const double*,  \
                               double*, double*, double*, double*, int*, int*,           \
                               const RatTab&);
LK_DECL(8)
LK_DECL(16)
LK_DECL(24)
LK_DECL(32)
LK_DECL(40)
LK_DECL(48)
LK_DECL(50)
LK_DECL(56)
LK_DECL(64)
#undef LK_DECL

int launch_tridiag_pair(hipStream_t st, int64_t np, const int32_t* perm, int KQ, int NV, int k,
                        int K, const LocDev& L, const StateDev& S, const VarsDev& V,
                        const ChunkDev& C, const DiagDev& D, double* B, const double* bvec,
                        double* tau, double* dd, double* ee, double* U, int* nvec,
                        int* status, const RatTab& R) {
  switch (KQ) {
    case 8: return launch_tridiag_pair_8(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    case 16: return launch_tridiag_pair_16(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    case 24: return launch_tridiag_pair_24(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    case 32: return launch_tridiag_pair_32(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    case 40: return launch_tridiag_pair_40(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    case 48: return launch_tridiag_pair_48(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    case 50: return launch_tridiag_pair_50(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    case 56: return launch_tridiag_pair_56(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    case 64: return launch_tridiag_pair_64(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee, U, nvec, status, R);
    default: return 0;
  }
}

}  // namespace lk
