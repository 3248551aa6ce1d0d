// BlockPool: a context's device and pinned blocks between the objects that use
// them (lsdg_internal.h).
#include "lsdg_internal.h"

namespace lsdg {

static size_t rounded(size_t bytes) { return (bytes + 4095) & ~(size_t)4095; }

hipError_t BlockPool::allocate(void** p, size_t bytes) {
  return host_ ? hipHostMalloc(p, bytes, hipHostMallocMapped) : hipMalloc(p, bytes);
}

void BlockPool::release(void* p) {
  if (host_) (void)hipHostFree(p);
  else (void)hipFree(p);
}

hipError_t BlockPool::take(void** p, size_t bytes) {
  *p = nullptr;
  bytes = rounded(bytes ? bytes : 1);
  std::lock_guard<std::mutex> lock(m_);
  auto it = idle_.lower_bound(bytes);
  if (it != idle_.end() && it->first - bytes <= bytes / 4) {
    *p = it->second;
    idleBytes_ -= it->first;
    live_[*p] = it->first;
    idle_.erase(it);
    return hipSuccess;
  }
  hipError_t e = allocate(p, bytes);
  if (e != hipSuccess && !idle_.empty()) {
    (void)hipGetLastError();
    for (auto& b : idle_) release(b.second);
    idle_.clear();
    idleBytes_ = 0;
    e = allocate(p, bytes);
  }
  if (e != hipSuccess) {
    *p = nullptr;
    return e;
  }
  live_[*p] = bytes;
  return hipSuccess;
}

void BlockPool::put(void* p) {
  if (!p) return;
  std::lock_guard<std::mutex> lock(m_);
  auto it = live_.find(p);
  if (it == live_.end()) return;
  const size_t bytes = it->second;
  live_.erase(it);
  if (idleBytes_ + bytes > limit_) {
    release(p);
    return;
  }
  idle_.emplace(bytes, p);
  idleBytes_ += bytes;
}

void BlockPool::trim() {
  std::lock_guard<std::mutex> lock(m_);
  for (auto& b : idle_) release(b.second);
  idle_.clear();
  idleBytes_ = 0;
}

}  // namespace lsdg
