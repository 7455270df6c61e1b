// Device memory of the library.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>

namespace sstg {

// Device memory that outlives the graph it was allocated for: allocating and
// freeing are the larger part of a short-lived graph's time (a hipFree waits
// for the device and unmaps, 0.25 ms and more each; loading a rMat scale-20
// graph and dropping it took 35 of them, 6.2 of 8.9 ms).  dev_free keeps a
// block for the next dev_alloc of its device that it fits (at most half again
// the size asked for), up to kDevKeep bytes in all; what is over goes back to
// HIP, and everything does when an allocation of this library fails and when
// the free memory is asked for.  The caller of dev_free has waited for the
// work that used the block: it may be handed to another stream at once.
// dev_release gives a block back to HIP in any case (waiting for the device,
// as hipFree does).  Blocks that dev_alloc did not make are passed on to
// hipFree.  dev_malloc is a hipMalloc that gives the kept blocks back and
// tries again before it fails, for memory that is not kept (freed with
// hipFree, dev_free or dev_release).  Any thread.
constexpr size_t kDevKeep = 4ull << 30;
hipError_t dev_malloc(void **out, size_t bytes);
hipError_t dev_alloc(void **out, size_t bytes, size_t *got = nullptr);
void dev_free(void *p);
void dev_release(void *p);
void dev_trim();
template <class T> hipError_t dev_alloc(T **out, size_t bytes) {
  void *p = nullptr;
  const hipError_t e = dev_alloc(&p, bytes, nullptr);
  *out = static_cast<T *>(p);
  return e;
}
template <class T> hipError_t dev_malloc(T **out, size_t bytes) {
  void *p = nullptr;
  const hipError_t e = dev_malloc(&p, bytes);
  *out = static_cast<T *>(p);
  return e;
}

}  // namespace sstg
