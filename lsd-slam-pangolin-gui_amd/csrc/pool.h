// Device and pinned host memory of the library: allocation, and the blocks that
// a context's objects give back (pool.cpp).
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <map>
#include <mutex>
#include <unordered_map>

namespace lsdg {

// Device memory, or pinned and host-mapped memory.  Where there is none left,
// every pool's idle blocks of that kind go back first.
hipError_t alloc_device(void** p, size_t bytes);
hipError_t alloc_pinned(void** p, size_t bytes);

// Device or pinned host blocks that a context's objects give back, kept for
// the next ones: allocating and freeing a frame's arrays cost 38 of the 63 us
// that making and destroying a 320x240 frame took, and a batch plan has eight
// device and four pinned blocks.  An idle block serves a request of at least
// four fifths of its size.  At most `limit` bytes stay idle: a block given back
// makes room by freeing the ones idle longest, so blocks of sizes no longer
// asked for don't keep the present ones out (2048x1536 frames made and
// destroyed beside an idle block of 236 MiB: 437 us each, now 121).  All of it
// is given back when an allocation of the process fails and with the context.  A block is given back only when no
// queued work of another stream than the context's touches it, and a pinned
// one when nothing queued does.  Nothing throws.
class BlockPool {
 public:
  BlockPool(bool host, size_t limit);
  BlockPool(const BlockPool&) = delete;
  BlockPool& operator=(const BlockPool&) = delete;
  ~BlockPool();
  template <class T>
  hipError_t get(T** p, size_t bytes) {
    void* q = nullptr;
    hipError_t e = take(&q, bytes);
    *p = static_cast<T*>(q);
    return e;
  }
  void put(void* p);  // null: nothing
  void trim();        // frees every idle block
  // trim() of every pool of one kind in the process; no pool's lock may be held
  static void trim_all(bool host);

 private:
  hipError_t take(void** p, size_t bytes);
  void release(void* p);
  const bool host_;
  const size_t limit_;
  BlockPool *next_ = nullptr, *prev_ = nullptr;  // all pools of the process
  std::mutex m_;
  struct Idle {
    void* p;
    unsigned long long since;
  };
  std::unordered_map<void*, size_t> live_;
  std::multimap<size_t, Idle> idle_;  // by size
  size_t idleBytes_ = 0;
  unsigned long long puts_ = 0;
};
constexpr size_t POOL_DEVICE_BYTES = (size_t)256 << 20;
constexpr size_t POOL_HOST_BYTES = (size_t)16 << 20;

}  // namespace lsdg
