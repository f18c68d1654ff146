// transform_row_kq72.hip -- k_row_tridiag and k_row_back for rows of 72
// (64 <= k <= 72); one instantiation per file keeps the build parallel.
#include "transform_row.h"

namespace lk {

void launch_row_tridiag_kq72(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                              double* bvec, double* tau, double* dd, double* ee) {
  launch_row_tridiag_kq<72>(st, nb, k, C, B, bvec, tau, dd, ee);
}

void launch_row_back_kq72(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                           double* bvec, const double* tau) {
  launch_row_back_kq<72>(st, nb, k, C, B, bvec, tau);
}

}  // namespace lk
