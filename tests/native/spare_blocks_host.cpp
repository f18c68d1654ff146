// Host build of umd-letkf_amd/csrc/spare_blocks.h for the CPU tests.
#include "../../umd-letkf_amd/csrc/spare_blocks.h"

#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <thread>
#include <vector>

using lk::SpareBlocks;

static std::vector<intptr_t> g_freed;
static void note(void* p) { g_freed.push_back((intptr_t)p); }
static std::atomic<long> g_live{0};
static void give(void* p) {
  std::free(p);
  --g_live;
}

extern "C" {
void* sb_new(int device) {
  SpareBlocks* s = new SpareBlocks(note);
  s->set_device(device);
  return s;
}
void sb_delete(void* s) { delete (SpareBlocks*)s; }
void sb_keep(void* s, intptr_t p, size_t size) { ((SpareBlocks*)s)->keep((void*)p, size); }
intptr_t sb_take(void* s, size_t least, size_t most, size_t* size) {
  return (intptr_t)((SpareBlocks*)s)->take(least, most, size);
}
size_t sb_bytes(void* s) { return ((SpareBlocks*)s)->bytes(); }
void sb_release(void* s) { ((SpareBlocks*)s)->release(); }
int sb_release_device(int device) { return SpareBlocks::release_device(device); }
size_t sb_most() { return SpareBlocks::kMost; }
int sb_count() { return SpareBlocks::kCount; }
// what was given back since the last call
int sb_freed(intptr_t* out, int n) {
  const int m = (int)g_freed.size();
  for (int i = 0; i < m && i < n; ++i) out[i] = g_freed[i];
  g_freed.clear();
  return m;
}
// threads with a handle each, and one that takes back what all of them keep;
// returns the blocks that were lost or given back twice
long sb_threads(int nthreads, int rounds) {
  std::atomic<bool> go{true};
  std::thread thief([&] { while (go) SpareBlocks::release_device(7); });
  std::vector<std::thread> ts;
  for (int t = 0; t < nthreads; ++t)
    ts.emplace_back([=] {
      SpareBlocks s(give);
      s.set_device(7);
      for (int i = 0; i < rounds; ++i) {
        size_t size = 1 + (size_t)(i * 37 + t) % 900, got = size;
        char* p = (char*)s.take(size, 2 * size, &got);
        if (!p) {
          p = (char*)std::malloc(size);
          ++g_live;
        }
        p[0] = p[got - 1] = (char)i;
        s.keep(p, got);
      }
    });
  for (auto& t : ts) t.join();
  go = false;
  thief.join();
  return g_live.load();
}
}
