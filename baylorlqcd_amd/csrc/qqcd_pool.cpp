// qqcd_pool.cpp -- see qqcd_pool.h.
#include "qqcd_pool.h"

#include <map>
#include <mutex>
#include <stdexcept>
#include <string>
#include <unordered_map>
#include <utility>
#include <vector>

#include "qqcd_internal.h"

namespace qqcd {

namespace {

typedef std::pair<int, size_t> Key;  // device (-1: pinned host memory) and rounded size

struct Pool {
  std::mutex mu;
  std::map<Key, std::vector<void *>> idle;
  std::unordered_map<void *, Key> live;
  size_t idle_bytes = 0, cap = 0;
};

// never destroyed: buffers may be returned by objects of static storage
// duration, and the runtime's own teardown releases what is left
Pool &pool() {
  static Pool *p = new Pool;
  return *p;
}

size_t rounded(size_t bytes) {
  const size_t q = bytes >= (size_t(1) << 20) ? size_t(2) << 20 : size_t(4) << 10;
  return (bytes + q - 1) / q * q;
}

void release(const Key &k, void *p) {
  if (k.first < 0) (void)hipHostFree(p);
  else (void)hipFree(p);
}

void drop_idle(Pool &P) {
  for (auto &e : P.idle)
    for (void *p : e.second) release(e.first, p);
  P.idle.clear();
  P.idle_bytes = 0;
}

void *take(int dev, size_t bytes) {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  const Key k(dev, rounded(bytes ? bytes : 1));
  void *p = nullptr;
  auto it = P.idle.find(k);
  if (it != P.idle.end() && !it->second.empty()) {
    p = it->second.back();
    it->second.pop_back();
    P.idle_bytes -= k.second;
  } else {
    auto get = [&]() { return dev < 0 ? hipHostMalloc(&p, k.second, hipHostMallocDefault) : hipMalloc(&p, k.second); };
    hipError_t e = get();
    if (e == hipErrorOutOfMemory && P.idle_bytes > 0) {
      (void)hipGetLastError();
      (void)hipDeviceSynchronize();
      drop_idle(P);
      e = get();
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      throw std::runtime_error(std::string("allocation of ") + std::to_string(k.second) + " bytes: " +
                               hipGetErrorString(e));
    }
  }
  P.live[p] = k;
  return p;
}

void give(void *p) {
  if (!p) return;
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  auto it = P.live.find(p);
  if (it == P.live.end()) return;
  const Key k = it->second;
  P.live.erase(it);
  if (!P.cap) {
    size_t free_b = 0, total = 0;
    P.cap = hipMemGetInfo(&free_b, &total) == hipSuccess && total ? total / 4 : size_t(1) << 30;
  }
  if (P.idle_bytes + k.second > P.cap) {
    release(k, p);
    return;
  }
  P.idle[k].push_back(p);
  P.idle_bytes += k.second;
}

}  // namespace

void *pool_alloc(size_t bytes) {
  int dev = 0;
  QQCD_HIP(hipGetDevice(&dev));
  return take(dev, bytes);
}
void pool_free(void *p) { give(p); }
void *pool_alloc_host(size_t bytes) { return take(-1, bytes); }
void pool_free_host(void *p) {
  if (!p) return;
  (void)hipDeviceSynchronize();
  give(p);
}

void pool_trim() {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  if (P.idle.empty()) return;
  (void)hipDeviceSynchronize();
  drop_idle(P);
}

}  // namespace qqcd
