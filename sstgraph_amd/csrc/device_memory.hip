// Device memory kept from dropped graphs for the next ones (host code only).
#include "device_memory.hpp"

#include <mutex>
#include <unordered_map>
#include <vector>

namespace sstg {

namespace {
struct DevBlock {
  void *p;
  size_t bytes;
  int dev;
};
// Never destroyed: graphs may be dropped while the process's statics go.
struct DevCache {
  std::mutex mu;
  std::vector<DevBlock> idle;                   // newest last
  std::unordered_map<void *, DevBlock> in_use;  // blocks dev_alloc handed out
  size_t idle_bytes = 0;
};
DevCache &dev_cache() {
  static DevCache *c = new DevCache();
  return *c;
}
}  // namespace

hipError_t dev_malloc(void **out, size_t bytes) {
  hipError_t e = hipMalloc(out, bytes ? bytes : 1);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    dev_trim();
    e = hipMalloc(out, bytes ? bytes : 1);
  }
  if (e != hipSuccess) *out = nullptr;
  return e;
}

hipError_t dev_alloc(void **out, size_t bytes, size_t *got) {
  DevCache &c = dev_cache();
  *out = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (!bytes) bytes = 1;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    size_t best = c.idle.size();
    for (size_t i = 0; i < c.idle.size(); i++) {
      const DevBlock &b = c.idle[i];
      if (b.dev == dev && b.bytes >= bytes && b.bytes - bytes <= bytes / 2 &&
          (best == c.idle.size() || b.bytes < c.idle[best].bytes))
        best = i;
    }
    if (best < c.idle.size()) {
      const DevBlock b = c.idle[best];
      c.idle.erase(c.idle.begin() + (ptrdiff_t)best);
      c.idle_bytes -= b.bytes;
      c.in_use[b.p] = b;
      *out = b.p;
      if (got) *got = b.bytes;
      return hipSuccess;
    }
  }
  e = dev_malloc(out, bytes);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(c.mu);
  c.in_use[*out] = DevBlock{*out, bytes, dev};
  if (got) *got = bytes;
  return hipSuccess;
}

void dev_free(void *p) {
  if (!p) return;
  DevCache &c = dev_cache();
  std::vector<void *> back;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto it = c.in_use.find(p);
    if (it == c.in_use.end() || it->second.bytes > kDevKeep / 2) {
      if (it != c.in_use.end()) c.in_use.erase(it);
      back.push_back(p);
    } else {
      c.idle.push_back(it->second);
      c.idle_bytes += it->second.bytes;
      c.in_use.erase(it);
      while (c.idle_bytes > kDevKeep) {  // the oldest first
        back.push_back(c.idle.front().p);
        c.idle_bytes -= c.idle.front().bytes;
        c.idle.erase(c.idle.begin());
      }
    }
  }
  for (void *q : back) (void)hipFree(q);
}

void dev_release(void *p) {
  if (!p) return;
  DevCache &c = dev_cache();
  {
    std::lock_guard<std::mutex> lk(c.mu);
    c.in_use.erase(p);
  }
  (void)hipFree(p);
}

void dev_trim() {
  DevCache &c = dev_cache();
  std::vector<DevBlock> back;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    back.swap(c.idle);
    c.idle_bytes = 0;
  }
  for (const DevBlock &b : back) (void)hipFree(b.p);
}

}  // namespace sstg
