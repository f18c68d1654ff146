// Host build of the search's short distance and weight (det_math.h), so that a
// CPU test can compare them with the full ones.
#include "../../umd-letkf_amd/csrc/det_math.h"

extern "C" {
// counts: values where the short form is sure but differs, and where it is not sure
void sfh_dist(long n, const double* c2, long* wrong, long* unsure) {
  for (long i = 0; i < n; ++i) {
    bool sure = false;
    const float d = dm::dist_fast(c2[i], &sure);
    if (!sure) ++*unsure;
    else if (d != dm::dist(c2[i])) ++*wrong;
  }
}
// a sure 0 stands for every weight that is not above 1e-4
void sfh_gc(long n, const float* z, const float* L, long* wrong, long* unsure) {
  for (long i = 0; i < n; ++i) {
    bool sure = false;
    const float w = dm::gc_fast(z[i], dm::gc_scale(L[i]), &sure), full = dm::gc(z[i], L[i]);
    if (!sure) ++*unsure;
    else if (w != full && !(w == 0.0f && !(full > 1.0e-4f))) ++*wrong;
  }
}
}
