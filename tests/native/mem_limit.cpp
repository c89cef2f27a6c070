// Test infrastructure: stands in front of the HIP runtime's allocators, so
// that a test can run the library as on a device with less memory or a host
// without pinned memory.  Loaded before the library, with its symbols global.
#include <dlfcn.h>

#include <atomic>
#include <cstddef>
#include <mutex>
#include <unordered_map>

namespace {
std::mutex mu;
std::unordered_map<void*, size_t> blocks;
size_t live = 0, peak = 0, limit = ~(size_t)0;
long calls = 0;
std::atomic<int> pinned_ok{1};

template <class F>
F real(const char* name) {
  return (F)dlsym(RTLD_NEXT, name);
}
}  // namespace

extern "C" {

// Bytes that live blocks may hold together from now on.
void nfm_limit(size_t bytes) { limit = bytes; }
void nfm_pinned(int ok) { pinned_ok = ok; }
size_t nfm_live() { return live; }
size_t nfm_peak() { return peak; }
long nfm_calls() { return calls; }
void nfm_reset_peak() { peak = live; }

int hipMalloc(void** p, size_t size) {
  static const auto f = real<int (*)(void**, size_t)>("hipMalloc");
  std::lock_guard<std::mutex> lock(mu);
  ++calls;
  // refused as the runtime refuses what no device has
  if (size > limit || live > limit - size) return f(p, (size_t)1 << 60);
  const int e = f(p, size);
  if (e == 0) {
    blocks[*p] = size;
    live += size;
    if (live > peak) peak = live;
  }
  return e;
}

int hipFree(void* p) {
  static const auto f = real<int (*)(void*)>("hipFree");
  std::lock_guard<std::mutex> lock(mu);
  auto it = blocks.find(p);
  if (it != blocks.end()) {
    live -= it->second;
    blocks.erase(it);
  }
  return f(p);
}

int hipHostMalloc(void** p, size_t size, unsigned flags) {
  static const auto f = real<int (*)(void**, size_t, unsigned)>("hipHostMalloc");
  if (!pinned_ok) return 2;  // hipErrorOutOfMemory
  return f(p, size, flags);
}

}  // extern "C"
