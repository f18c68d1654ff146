// spare_blocks.h -- the device blocks that a handle keeps between its calls
// (host code, no HIP types: tested without a GPU).
#pragma once

#include <algorithm>
#include <cstddef>
#include <mutex>

namespace lk {

// Blocks of one handle that no call uses, at most kMost bytes and kCount of
// them: the oldest leave first, so a size that is never asked for again makes
// room.  A thread whose allocation failed may take back what every handle on
// its device keeps (release_device), so all of them are known to one list
// under one lock; blocks are given to `release` with the lock let go, since a
// release may wait for the device.
class SpareBlocks {
 public:
  static constexpr size_t kMost = 1ull << 30;
  static constexpr int kCount = 64;
  typedef void (*Release)(void*);

  explicit SpareBlocks(Release f) : free_(f) {
    std::lock_guard<std::mutex> g(m_);
    next_ = head_;
    head_ = this;
  }
  ~SpareBlocks() {
    release();
    std::lock_guard<std::mutex> g(m_);
    SpareBlocks** at = &head_;
    while (*at != this) at = &(*at)->next_;
    *at = next_;
  }
  SpareBlocks(const SpareBlocks&) = delete;
  SpareBlocks& operator=(const SpareBlocks&) = delete;

  void set_device(int device) {
    std::lock_guard<std::mutex> g(m_);
    device_ = device;
  }
  size_t bytes() const {
    std::lock_guard<std::mutex> g(m_);
    return bytes_;
  }

  // the smallest block of least .. most bytes (*size its own), or nullptr
  void* take(size_t least, size_t most, size_t* size) {
    std::lock_guard<std::mutex> g(m_);
    int at = -1;
    for (int i = 0; i < n_; ++i)
      if (b_[i].size >= least && b_[i].size <= most && (at < 0 || b_[i].size < b_[at].size)) at = i;
    if (at < 0) return nullptr;
    const Block got = b_[at];
    drop(at);
    *size = got.size;
    return got.p;
  }

  // p (size bytes) is not used any more
  void keep(void* p, size_t size) {
    if (size > kMost) {
      free_(p);
      return;
    }
    Block out[kCount];
    int n = 0;
    {
      std::lock_guard<std::mutex> g(m_);
      while (n_ > 0 && (n_ == kCount || bytes_ + size > kMost)) {
        out[n++] = b_[0];
        drop(0);
      }
      b_[n_++] = Block{p, size, free_};
      bytes_ += size;
    }
    for (int i = 0; i < n; ++i) free_(out[i].p);
  }

  // everything kept goes back to the device
  void release() {
    Block b;
    while (pop([this](const SpareBlocks& s) { return &s == this; }, &b)) free_(b.p);
  }

  // and what the other handles on a device keep; false if there was nothing
  static bool release_device(int device) {
    bool any = false;
    Block b;
    while (pop([device](const SpareBlocks& s) { return s.device_ == device; }, &b)) {
      b.owner(b.p);
      any = true;
    }
    return any;
  }

 private:
  struct Block {
    void* p;
    size_t size;
    Release owner;
  };
  // the last block of the first handle that is meant and keeps one
  template <typename Meant>
  static bool pop(Meant&& meant, Block* out) {
    std::lock_guard<std::mutex> g(m_);
    for (SpareBlocks* s = head_; s; s = s->next_)
      if (s->n_ > 0 && meant(*s)) {
        *out = s->b_[s->n_ - 1];
        s->drop(s->n_ - 1);
        return true;
      }
    return false;
  }
  void drop(int at) {
    bytes_ -= b_[at].size;
    std::copy(b_ + at + 1, b_ + n_, b_ + at);
    --n_;
  }

  static inline std::mutex m_;
  static inline SpareBlocks* head_ = nullptr;
  SpareBlocks* next_ = nullptr;
  Release free_;
  int device_ = -1;
  Block b_[kCount];
  int n_ = 0;
  size_t bytes_ = 0;
};

}  // namespace lk
