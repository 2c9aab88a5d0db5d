// qqcd_pool.h -- device and pinned host buffers kept between calls.
//
// Every solve, operator call and field transfer needs a handful to several
// hundred temporary fields of a few recurring sizes.  hipMalloc + hipFree of
// one costs 100-300 us (hipFree waits for the device and unmaps), which for
// the 50-300 fields of a solve was 60-90 ms: 30% of a 24-source noise loop
// and half of an FP32 mixed solve at 16^3x32.  A freed buffer therefore goes
// to a free list of its size and the next request of that size takes it.
//
//  * Order: a buffer may be freed while work on it is still queued on the
//    context's stream; its next user queues on that same stream (the library
//    has one) or on the null stream, which waits for it.  A pinned buffer's next
//    user is the host, so returning one waits for the device.
//  * Bounds: the free lists hold at most a quarter of the device's memory and 1
//    GiB of pinned memory (beyond that the buffers given back longest ago are
//    released, so that a program that changes its sizes keeps its current ones);
//    a failed hipMalloc releases them and tries again; qqcd_init and
//    qqcd_finalize release them all.
//  * Contents are undefined: a caller that needs zeros clears the buffer.
//  * Calls from several threads are serialised by a mutex.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

namespace qqcd {

void *pool_alloc(size_t bytes);
void pool_free(void *p);
void *pool_alloc_host(size_t bytes);  // pinned
void pool_free_host(void *p);
void pool_trim();  // releases every free buffer (waits for the device first)

// hipMalloc for a buffer that outlives calls (freed by hipFree): idle buffers
// are released where the card has no room for it
hipError_t device_malloc_bytes(void **p, size_t bytes);
template <typename T> hipError_t device_malloc(T **p, size_t bytes) {
  return device_malloc_bytes(reinterpret_cast<void **>(p), bytes);
}

template <typename T> void pool_get(T **p, size_t bytes) { *p = static_cast<T *>(pool_alloc(bytes)); }

// The buffers of one object, returned with it, also where its constructor fails
// halfway.
class PoolSet {
 public:
  PoolSet() = default;
  ~PoolSet() {
    for (void *p : device) pool_free(p);
    for (void *p : pinned) pool_free_host(p);
  }
  PoolSet(const PoolSet &) = delete;
  PoolSet &operator=(const PoolSet &) = delete;
  template <typename T> void get(T **p, size_t bytes) {
    device.reserve(device.size() + 1);
    device.push_back(*p = static_cast<T *>(pool_alloc(bytes)));
  }
  template <typename T> void get_host(T **p, size_t bytes) {
    pinned.reserve(pinned.size() + 1);
    pinned.push_back(*p = static_cast<T *>(pool_alloc_host(bytes)));
  }

 private:
  std::vector<void *> device, pinned;
};

}  // namespace qqcd
