// Allocation and BlockPool (pool.h).  Locks: the list of pools before a pool's
// own; allocations run under neither, as a failed one trims every pool.
#include "pool.h"

#include <exception>

namespace lsdg {

static std::mutex g_poolsMutex;
static BlockPool* g_pools = nullptr;

static size_t rounded(size_t bytes) { return (bytes + 4095) & ~(size_t)4095; }

static hipError_t allocate(bool host, void** p, size_t bytes) {
  const auto once = [&] { return host ? hipHostMalloc(p, bytes, hipHostMallocMapped) : hipMalloc(p, bytes); };
  hipError_t e = once();
  if (e != hipSuccess) {
    (void)hipGetLastError();
    BlockPool::trim_all(host);
    e = once();
  }
  if (e != hipSuccess) *p = nullptr;
  return e;
}

hipError_t alloc_device(void** p, size_t bytes) { return allocate(false, p, bytes); }
hipError_t alloc_pinned(void** p, size_t bytes) { return allocate(true, p, bytes); }

BlockPool::BlockPool(bool host, size_t limit) : host_(host), limit_(limit) {
  std::lock_guard<std::mutex> lock(g_poolsMutex);
  next_ = g_pools;
  if (next_) next_->prev_ = this;
  g_pools = this;
}

BlockPool::~BlockPool() {
  {
    std::lock_guard<std::mutex> lock(g_poolsMutex);
    (prev_ ? prev_->next_ : g_pools) = next_;
    if (next_) next_->prev_ = prev_;
  }
  trim();
}

void BlockPool::trim_all(bool host) {
  std::lock_guard<std::mutex> lock(g_poolsMutex);
  for (BlockPool* q = g_pools; q; q = q->next_)
    if (q->host_ == host) q->trim();
}

void BlockPool::release(void* p) {
  if (host_) (void)hipHostFree(p);
  else (void)hipFree(p);
}

hipError_t BlockPool::take(void** p, size_t bytes) {
  *p = nullptr;
  bytes = rounded(bytes ? bytes : 1);
  try {
    std::lock_guard<std::mutex> lock(m_);
    auto it = idle_.lower_bound(bytes);
    if (it != idle_.end() && it->first - bytes <= bytes / 4) {
      live_.emplace(it->second.p, it->first);
      *p = it->second.p;
      idleBytes_ -= it->first;
      idle_.erase(it);
      return hipSuccess;
    }
  } catch (const std::exception&) {
    return hipErrorOutOfMemory;  // of the host, for the pool's own record
  }
  hipError_t e = allocate(host_, p, bytes);
  if (e != hipSuccess) return e;
  try {
    std::lock_guard<std::mutex> lock(m_);
    live_.emplace(*p, bytes);
  } catch (const std::exception&) {
    release(*p);
    *p = nullptr;
    return hipErrorOutOfMemory;
  }
  return hipSuccess;
}

void BlockPool::put(void* p) {
  if (!p) return;
  std::lock_guard<std::mutex> lock(m_);
  auto it = live_.find(p);
  if (it == live_.end()) return;
  const size_t bytes = it->second;
  live_.erase(it);
  if (bytes <= limit_) {
    try {
      idle_.emplace(bytes, Idle{p, puts_++});
      idleBytes_ += bytes;
      p = nullptr;
    } catch (const std::exception&) {  // no record of it: freed
    }
  }
  if (p) release(p);
  while (idleBytes_ > limit_) {
    auto oldest = idle_.begin();
    for (auto b = idle_.begin(); b != idle_.end(); ++b)
      if (b->second.since < oldest->second.since) oldest = b;
    release(oldest->second.p);
    idleBytes_ -= oldest->first;
    idle_.erase(oldest);
  }
}

void BlockPool::trim() {
  std::lock_guard<std::mutex> lock(m_);
  for (auto& b : idle_) release(b.second.p);
  idle_.clear();
  idleBytes_ = 0;
}

}  // namespace lsdg
