// qqcd_pool.cpp -- see qqcd_pool.h.
#include "qqcd_pool.h"

#include <cstdint>
#include <deque>
#include <map>
#include <mutex>
#include <stdexcept>
#include <string>
#include <unordered_map>
#include <utility>

#include "qqcd_internal.h"

namespace qqcd {

namespace {

typedef std::pair<int, size_t> Key;  // device (-1: pinned host memory) and rounded size

// the free lists of device or of pinned memory; the newest of a size is at the back
struct Idle {
  std::map<Key, std::deque<std::pair<uint64_t, void *>>> lists;
  size_t bytes = 0, cap = 0;
};

struct Pool {
  std::mutex mu;
  Idle device, pinned;
  std::unordered_map<void *, Key> live;
  uint64_t returned = 0;  // buffers given back so far: what orders them
  Idle &of(const Key &k) { return k.first < 0 ? pinned : device; }
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

void drop_idle(Idle &I) {
  for (auto &e : I.lists)
    for (auto &b : e.second) release(e.first, b.second);
  I.lists.clear();
  I.bytes = 0;
}

// releases the buffers given back longest ago until `bytes` more fit
void make_room(Idle &I, size_t bytes) {
  while (I.bytes + bytes > I.cap) {
    auto old = I.lists.end();
    for (auto it = I.lists.begin(); it != I.lists.end(); ++it)
      if (old == I.lists.end() || it->second.front().first < old->second.front().first) old = it;
    if (old == I.lists.end()) return;
    release(old->first, old->second.front().second);
    I.bytes -= old->first.second;
    old->second.pop_front();
    if (old->second.empty()) I.lists.erase(old);
  }
}

void *take(int dev, size_t bytes) {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  const Key k(dev, rounded(bytes ? bytes : 1));
  void *p = nullptr;
  Idle &I = P.of(k);
  auto it = I.lists.find(k);
  if (it != I.lists.end()) {
    p = it->second.back().second;
    it->second.pop_back();
    if (it->second.empty()) I.lists.erase(it);
    I.bytes -= k.second;
  } else {
    auto get = [&]() { return dev < 0 ? hipHostMalloc(&p, k.second, hipHostMallocDefault) : hipMalloc(&p, k.second); };
    hipError_t e = get();
    if (e == hipErrorOutOfMemory && I.bytes > 0) {
      (void)hipGetLastError();
      (void)hipDeviceSynchronize();
      drop_idle(I);
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
  Idle &I = P.of(k);
  if (!I.cap) {
    size_t free_b = 0, total = 0;
    const bool known = k.first >= 0 && hipMemGetInfo(&free_b, &total) == hipSuccess && total;
    I.cap = known ? total / 4 : size_t(1) << 30;
  }
  if (k.second > I.cap) {
    release(k, p);
    return;
  }
  make_room(I, k.second);
  I.lists[k].emplace_back(P.returned++, p);
  I.bytes += k.second;
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

hipError_t device_malloc_bytes(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();  // the caller reports it, no later launch
    Pool &P = pool();
    std::lock_guard<std::mutex> lock(P.mu);
    if (P.device.lists.empty()) return e;
    (void)hipDeviceSynchronize();
    drop_idle(P.device);
    e = hipMalloc(p, bytes);
    if (e != hipSuccess) (void)hipGetLastError();
  }
  return e;
}

void pool_trim() {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  if (P.device.lists.empty() && P.pinned.lists.empty()) return;
  (void)hipDeviceSynchronize();
  drop_idle(P.device);
  drop_idle(P.pinned);
}

}  // namespace qqcd
