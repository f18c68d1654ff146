// transform_row_kq96.hip -- k_row_tridiag and k_row_back for rows of 96
// (89 <= k <= 96); one instantiation per file keeps the build parallel.
#include "transform_row.h"

namespace lk {

void launch_row_tridiag_kq96(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                              double* bvec, double* tau, double* dd, double* ee) {
  launch_row_tridiag_kq<96>(st, nb, k, C, B, bvec, tau, dd, ee);
}

void launch_row_back_kq96(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                           double* bvec, const double* tau) {
  launch_row_back_kq<96>(st, nb, k, C, B, bvec, tau);
}

}  // namespace lk
