// Cache of device blocks (see devmem.h).
#include "devmem.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>

namespace mmsb {

namespace {
struct DevCache {
  std::mutex mu;
  std::multimap<std::pair<int, size_t>, void*> kept;              // (device, bytes) -> block
  std::unordered_map<void*, std::pair<int, size_t>> live;         // blocks handed out
  size_t bytes = 0;                                               // of the kept blocks
};

DevCache& dev_cache() {
  static DevCache* c = new DevCache;  // not destroyed: contexts may outlive static destruction
  return *c;
}

void drop(DevCache& c) {
  for (auto& b : c.kept) (void)hipFree(b.second);
  c.kept.clear();
  c.bytes = 0;
}

// hipMalloc, once more without the kept blocks if it fails.
hipError_t malloc_or_drop(DevCache& c, void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess && !c.kept.empty()) {
    (void)hipGetLastError();
    drop(c);
    e = hipMalloc(p, bytes);
  }
  return e;
}
}  // namespace

hipError_t dev_alloc(void** p, size_t bytes) {
  *p = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  DevCache& c = dev_cache();
  std::lock_guard<std::mutex> lock(c.mu);
  // the smallest kept block that is large enough, by at most an eighth and a page
  auto it = c.kept.lower_bound({dev, bytes});
  if (it != c.kept.end() && it->first.first == dev && it->first.second <= bytes + bytes / 8 + 4096) {
    *p = it->second;
    c.live[*p] = it->first;
    c.bytes -= it->first.second;
    c.kept.erase(it);
    return hipSuccess;
  }
  e = malloc_or_drop(c, p, bytes);
  if (e == hipSuccess) c.live[*p] = {dev, bytes};
  return e;
}

hipError_t dev_malloc(void** p, size_t bytes) {
  *p = nullptr;
  DevCache& c = dev_cache();
  std::lock_guard<std::mutex> lock(c.mu);
  return malloc_or_drop(c, p, bytes);
}

void dev_free(void* p) {
  if (!p) return;
  DevCache& c = dev_cache();
  std::lock_guard<std::mutex> lock(c.mu);
  auto it = c.live.find(p);
  if (it == c.live.end()) return;
  const std::pair<int, size_t> b = it->second;
  c.live.erase(it);
  if (c.bytes + b.second <= kDevCacheBytes) {
    c.kept.emplace(b, p);
    c.bytes += b.second;
  } else {
    (void)hipFree(p);
  }
}

void dev_release(void* p) {
  if (!p) return;
  DevCache& c = dev_cache();
  {
    std::lock_guard<std::mutex> lock(c.mu);
    if (c.live.erase(p) == 0) return;
  }
  (void)hipFree(p);
}

size_t dev_cached_bytes() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  DevCache& c = dev_cache();
  std::lock_guard<std::mutex> lock(c.mu);
  size_t n = 0;
  for (auto& b : c.kept) n += b.first.first == dev ? b.first.second : 0;
  return n;
}

void release_device_cache() {
  DevCache& c = dev_cache();
  std::lock_guard<std::mutex> lock(c.mu);
  drop(c);
}

}  // namespace mmsb
