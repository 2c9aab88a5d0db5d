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

// the lists are full of buffers of one size: a program that goes on with another gets its own back all the same, and
// the bound (a quarter of the card) holds
int other_size() {
  std::vector<void *> a;
  for (int i = 0; i < 8; i++) a.push_back(pool_alloc(2 * MB));
  for (void *p : a) pool_free(p);
  EXPECT(used == 16 * MB);
  for (int i = 0; i < 5; i++) {
    void *p = pool_alloc(4 * MB), *q = pool_alloc(4 * MB);
    pool_free(p);
    pool_free(q);
    EXPECT(used <= 16 * MB);
  }
  EXPECT(mallocs == 8 + 2);
  // the ones given back longest ago went: what is left of the first size is kept
  EXPECT(used == 16 * MB && frees == 4);
  // a buffer larger than the bound is not kept
  void *big = pool_alloc(20 * MB);
  pool_free(big);
  EXPECT(used <= 16 * MB);
  pool_trim();
  EXPECT(used == 0);
  return 0;
}

// pinned memory is the host's: it takes nothing of the card's share, and has a bound of its own
int pinned_share() {
  void *h = pool_alloc_host(15 * MB);
  pool_free_host(h);
  void *a = pool_alloc(8 * MB);
  pool_free(a);
  EXPECT(used == 8 * MB);
  EXPECT(pool_alloc(8 * MB) == a);
  std::vector<void *> v;
  for (int i = 0; i < 100; i++) v.push_back(pool_alloc_host(16 * MB));
  for (void *p : v) pool_free_host(p);
  EXPECT(pinned <= 1024 * MB);
  pool_trim();
  EXPECT(pinned == 0);
  return 0;
}

// a buffer that is not pooled gets the memory that idle ones hold
int unpooled() {
  for (int i = 0; i < 4; i++) {
    void *p = pool_alloc((2 + 2 * i) * MB);
    pool_free(p);
  }
  EXPECT(used > 0);
  void *p = nullptr;
  EXPECT(device_malloc(&p, 60 * MB) == hipSuccess);
  EXPECT(used == 60 * MB);
  double *q = nullptr;
  EXPECT(device_malloc(&q, 10 * MB) == hipErrorOutOfMemory);
  EXPECT(hipFree(p) == hipSuccess && used == 0);
  return 0;
}

// an object whose constructor fails returns what it has got so far
int half_built() {
  struct Object {
    PoolSet bufs;
    double *a = nullptr, *b = nullptr, *c = nullptr;
    Object() {
      bufs.get(&a, 2 * MB);
      bufs.get_host(&b, 2 * MB);
      bufs.get(&c, 100 * MB);
    }
  };
  bool thrown = false;
  try {
    Object o;
  } catch (const std::runtime_error &) {
    thrown = true;
  }
  EXPECT(thrown);
  pool_trim();
  EXPECT(used == 0 && pinned == 0);
  return 0;
}

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "pinned_wait") return pinned_wait();
  if (what == "other_size") return other_size();
  if (what == "pinned_share") return pinned_share();
  if (what == "unpooled") return unpooled();
  if (what == "half_built") return half_built();
  std::printf("no such check\n");
  return 2;
}
