// transform_row_kq88.hip -- k_row_tridiag and k_row_back for rows of 88
// (81 <= k <= 88); one instantiation per file keeps the build parallel.
#include "transform_row.h"

namespace lk {

void launch_row_tridiag_kq88(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                              double* bvec, double* tau, double* dd, double* ee) {
  launch_row_tridiag_kq<88>(st, nb, k, C, B, bvec, tau, dd, ee);
}

void launch_row_back_kq88(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                           double* bvec, const double* tau) {
  launch_row_back_kq<88>(st, nb, k, C, B, bvec, tau);
}

}  // namespace lk
