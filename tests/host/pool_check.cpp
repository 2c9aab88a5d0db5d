// The buffer pool (baylorlqcd_amd/csrc/qqcd_pool.cpp) on a runtime of this file's own: a card of `total` bytes that
// counts what is asked of it.  Prints the first expectation that does not hold and returns 1.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <stdexcept>
#include <string>
#include <vector>

#include "qqcd_pool.h"

namespace {
constexpr size_t MB = size_t(1) << 20;
size_t total = 64 * MB, used = 0, pinned = 0;
int mallocs = 0, frees = 0, waits = 0;
std::map<void *, size_t> sizes;
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  mallocs++;
  if (used + n > total) return hipErrorOutOfMemory;
  used += n;
  *p = std::malloc(16);
  sizes[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  frees++;
  used -= sizes.at(p);
  sizes.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  mallocs++;
  pinned += n;
  *p = std::malloc(16);
  sizes[*p] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  frees++;
  pinned -= sizes.at(p);
  sizes.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = total - used;
  *t = total;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  waits++;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
}

#define EXPECT(x)                                        \
  do {                                                   \
    if (!(x)) {                                          \
      std::printf("line %d: %s\n", __LINE__, #x);        \
      return 1;                                          \
    }                                                    \
  } while (0)

using namespace qqcd;

// a pinned buffer may be the target of copies still queued when it is given back: the device is waited for before
// anyone else gets it
int pinned_wait() {
  void *a = pool_alloc_host(4096);
  const int before = waits;
  pool_free_host(a);
  EXPECT(waits > before);
  EXPECT(pool_alloc_host(4096) == a);
  return 0;
}

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "pinned_wait") return pinned_wait();
  std::printf("no such check\n");
  return 2;
}
