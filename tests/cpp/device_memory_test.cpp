// csrc/device_memory.hip over a device of fixed size that exists only here:
// the HIP calls it makes are the functions below.  Prints "ok" and exits 0.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "device_memory.hpp"

namespace {
size_t capacity, used;
int frees;
std::map<void *, size_t> blocks;
uintptr_t next_address = 1 << 20;

void check(bool ok, const char *what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::exit(1);
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t bytes) {
  if (used + bytes > capacity) return hipErrorOutOfMemory;
  *p = reinterpret_cast<void *>(next_address);
  next_address += 4096;
  used += blocks[*p] = bytes;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  auto it = blocks.find(p);
  check(it != blocks.end(), "only live blocks are freed");
  used -= it->second;
  frees++;
  blocks.erase(it);
  return hipSuccess;
}
hipError_t hipGetDevice(int *dev) {
  *dev = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
}

int main() {
  using namespace sstg;
  const size_t mib = 1 << 20;
  capacity = 64 * mib;
  char *a = nullptr, *b = nullptr, *c = nullptr;
  check(dev_alloc(&a, 40 * mib) == hipSuccess, "first block");
  dev_free(a);
  check(frees == 0 && used == 40 * mib, "a dropped block is kept");
  check(dev_alloc(&b, 40 * mib) == hipSuccess && b == a, "and used again");
  // memory in use is not taken
  check(dev_malloc(&c, 40 * mib) == hipErrorOutOfMemory && !c, "no room");
  dev_free(b);
  check(dev_malloc(&c, 40 * mib) == hipSuccess && frees == 1,
        "dev_malloc takes the kept block's room");
  check(dev_alloc(&b, 40 * mib) == hipErrorOutOfMemory && !b, "no room again");
  dev_release(c);
  check(used == 0, "dev_release gives back");
  // dev_alloc too, where no kept block fits
  check(dev_alloc(&a, 10 * mib) == hipSuccess, "small block");
  dev_free(a);
  check(dev_alloc(&a, 60 * mib) == hipSuccess && used == 60 * mib,
        "dev_alloc takes the kept block's room");
  dev_free(a);
  dev_trim();
  check(used == 0 && blocks.empty(), "dev_trim gives all back");
  // what is kept is bounded
  capacity = 4 * kDevKeep;
  char *many[16];
  for (char *&p : many)
    check(dev_alloc(&p, kDevKeep / 4) == hipSuccess, "many blocks");
  for (char *p : many) dev_free(p);
  check(used == kDevKeep, "no more than kDevKeep is kept");
  check(dev_alloc(&a, kDevKeep) == hipSuccess, "a large block");
  dev_free(a);
  check(used == kDevKeep, "blocks over half of kDevKeep are not kept");
  check(dev_malloc(&a, 0) == hipSuccess && a, "no bytes: a block of its own");
  dev_free(a);
  std::puts("ok");
  return 0;
}
