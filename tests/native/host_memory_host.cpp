// Host build of umd-letkf_amd/csrc/host_memory.h for the CPU tests.
#include "../../umd-letkf_amd/csrc/host_memory.h"

extern "C" {
// locked allocations: npiece of (host address, device address, size)
const void* hm_locked_span(const char* p, size_t n, int npiece, const char* const* host,
                           char* const* dev, const size_t* size) {
  return lk::locked_span(p, n, [&](const void* q, lk::LockedPiece* out) {
    for (int i = 0; i < npiece; ++i) {
      const char* c = static_cast<const char*>(q);
      if (c < host[i] || c >= host[i] + size[i]) continue;
      *out = {dev[i] + (c - host[i]), dev[i], size[i]};
      return true;
    }
    return false;
  });
}
}
