// host_memory.h -- what the library decides about a caller's host memory
// (host code, no HIP types: the decisions are tested without a GPU).
#pragma once

#include <cstddef>

namespace lk {

// a piece of page-locked memory as the runtime knows it: the device's address
// of the pointer asked about, and the whole allocation it lies in
struct LockedPiece {
  char* dev = nullptr;
  const char* base = nullptr;   // the allocation's first byte, the device's address
  size_t size = 0;
};

// The device's address of n bytes at p, or nullptr where they are not one
// page-locked allocation's: a kernel that writes them must not leave it.
// piece(p, &out) asks the runtime and is false for memory that is not locked.
// (Both ends being locked is not enough: of two locked allocations with
// ordinary memory between them, addresses being the same for host and device,
// the ends lie as far apart on either side.)
template <typename Piece>
inline void* locked_span(const void* p, size_t n, Piece&& piece) {
  LockedPiece a;
  if (!p || n == 0 || !piece(p, &a) || !a.dev || a.dev < a.base) return nullptr;
  const size_t at = (size_t)(a.dev - a.base);
  return at <= a.size && n <= a.size - at ? a.dev : nullptr;
}

}  // namespace lk
