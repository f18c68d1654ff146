// transform_row_kq80.hip -- k_row_tridiag and k_row_back for rows of 80
// (73 <= k <= 80); one instantiation per file keeps the build parallel.
#include "transform_row.h"

namespace lk {

void launch_row_tridiag_kq80(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                              double* bvec, double* tau, double* dd, double* ee) {
  launch_row_tridiag_kq<80>(st, nb, k, C, B, bvec, tau, dd, ee);
}

void launch_row_back_kq80(hipStream_t st, unsigned nb, int k, const ChunkDev& C, double* B,
                           double* bvec, const double* tau) {
  launch_row_back_kq<80>(st, nb, k, C, B, bvec, tau);
}

}  // namespace lk
