// tridiag_pair_kq56.hip -- one-problem tridiagonalization, rows of 56.
#include "tridiag_pair.h"

namespace lk {

int launch_tridiag_pair_56(hipStream_t st, int64_t np, const int32_t* perm, int NV, int k, int K,
                           const LocDev& L, const StateDev& S, const VarsDev& V,
                           const ChunkDev& C, const DiagDev& D, double* B, const double* bvec,
                           double* tau, double* dd, double* ee, double* U, int* nvec,
                           int* status, const RatTab& R) {
  return launch_tridiag_pair_kq<56>(st, np, perm, NV, k, K, L, S, V, C, D, B, bvec, tau, dd, ee,
                                     U, nvec, status, R);
}

}  // namespace lk
