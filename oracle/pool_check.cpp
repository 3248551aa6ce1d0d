// The library's block pool (csrc/pool.cpp) over an allocator that counts and
// can run out: reuse, its bound and what it keeps, giving idle blocks back to
// other pools and to plain allocations, failing allocations of the host's own
// memory, and blocks given back by other threads.  Host code only; prints "ok"
// per check.
#include "../lsd-slam-pangolin-gui_amd/csrc/pool.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <thread>
#include <vector>

namespace {
std::mutex g_m;
std::map<void*, size_t>* g_blocks;
size_t g_used = 0, g_capacity = (size_t)-1, g_allocations = 0;
thread_local long g_failNewIn = -1;  // >= 0: the operator new after this many throws

hipError_t take(void** p, size_t n) {
  std::lock_guard<std::mutex> lock(g_m);
  if (n > g_capacity - g_used) {
    *p = nullptr;
    return hipErrorOutOfMemory;
  }
  *p = std::malloc(n);
  (*g_blocks)[*p] = n;
  g_used += n;
  ++g_allocations;
  return hipSuccess;
}
hipError_t give(void* p) {
  std::lock_guard<std::mutex> lock(g_m);
  auto it = g_blocks->find(p);
  if (it == g_blocks->end()) {
    std::printf("freed twice\n");
    std::exit(1);
  }
  g_used -= it->second;
  g_blocks->erase(it);
  std::free(p);
  return hipSuccess;
}
void expect(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::exit(1);
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  const long f = g_failNewIn;
  g_failNewIn = -1;  // the counted failures are the pool's own records
  hipError_t e = take(p, n);
  g_failNewIn = f;
  return e;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipGetLastError() { return hipSuccess; }
}

void* operator new(size_t n) {
  if (g_failNewIn >= 0 && g_failNewIn-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

using lsdg::BlockPool;
constexpr size_t KB = 1024;

int main() {
  g_blocks = new std::map<void*, size_t>;
  {  // an idle block serves requests of four fifths of its size and more
    BlockPool a(false, 1000 * KB);
    void *p, *q, *r;
    expect(a.get(&p, 100 * KB) == hipSuccess, "get");
    a.put(p);
    a.put(nullptr);
    expect(a.get(&q, 80 * KB) == hipSuccess && q == p, "reuse of a larger block");
    a.put(q);
    expect(a.get(&q, 76 * KB) == hipSuccess && q != p, "a block is not given to a much smaller request");
    expect(a.get(&r, 104 * KB) == hipSuccess && r != p, "nor to a larger one");
    a.put(q);
    a.put(r);
  }
  expect(g_used == 0, "a pool gives its idle blocks back at its end");
  std::printf("ok\n");
  {  // at most `limit` bytes idle
    BlockPool a(true, 64 * KB);
    std::vector<void*> v(8);
    for (void*& p : v) expect(a.get(&p, 16 * KB) == hipSuccess, "get");
    for (void* p : v) a.put(p);
    expect(g_used == 64 * KB, "idle bytes are bounded");
    // the blocks in use now replace the ones idle longest, and are found again
    void* p;
    for (int k = 0; k < 5; ++k) {
      const size_t before = g_allocations;
      expect(a.get(&p, 40 * KB) == hipSuccess, "get");
      a.put(p);
      expect(g_allocations == before + (k == 0 ? 1 : 0), "a size in use is kept beside older blocks");
      expect(g_used <= 64 * KB, "idle bytes are bounded");
    }
    expect(a.get(&p, 16 * KB) == hipSuccess && g_used == 56 * KB, "the newest of the older blocks stayed");
    a.put(p);
    expect(a.get(&p, 100 * KB) == hipSuccess, "get");
    a.put(p);
    expect(g_used == 56 * KB, "a block over the limit is freed, and no other");
  }
  std::printf("ok\n");
  {  // idle blocks go back where another pool, or a plain allocation, finds no memory
    BlockPool a(false, 1000 * KB), b(false, 1000 * KB), h(true, 1000 * KB);
    void *p, *q, *s;
    g_capacity = 100 * KB;
    expect(a.get(&p, 60 * KB) == hipSuccess && h.get(&s, 20 * KB) == hipSuccess, "get");
    a.put(p);
    expect(b.get(&q, 70 * KB) == hipSuccess, "another pool's idle block goes back");
    b.put(q);
    h.put(s);
    expect(lsdg::alloc_device(&p, 80 * KB) == hipSuccess && g_used == 100 * KB, "a plain allocation");
    expect(lsdg::alloc_device(&q, 8 * KB) == hipErrorOutOfMemory && q == nullptr, "and its failure");
    expect(b.get(&q, 8 * KB) == hipErrorOutOfMemory && q == nullptr, "a pool's failure");
    expect(lsdg::alloc_pinned(&q, 8 * KB) == hipSuccess && g_used == 88 * KB, "pinned pools are their own kind");
    (void)hipFree(p);
    (void)hipHostFree(q);
    g_capacity = (size_t)-1;
  }
  expect(g_used == 0, "nothing is left");
  std::printf("ok\n");
  {  // the host's memory runs out for the pool's records: an error or a free, no exception, no leak
    BlockPool a(false, 1000 * KB);
    for (long k = 0; k < 3; ++k) {
      void *p, *q = nullptr;
      g_failNewIn = k;
      hipError_t e = a.get(&p, 16 * KB);
      g_failNewIn = -1;
      expect(e == hipSuccess ? p != nullptr : e == hipErrorOutOfMemory && p == nullptr, "get without a record");
      if (e != hipSuccess) expect(a.get(&p, 16 * KB) == hipSuccess, "get");
      g_failNewIn = k;
      a.put(p);
      g_failNewIn = -1;
      g_failNewIn = k;
      e = a.get(&q, 16 * KB);
      g_failNewIn = -1;
      expect((e == hipSuccess) == (q != nullptr), "get of an idle block without a record");
      a.put(q);
    }
  }
  expect(g_used == 0, "nothing is left");
  std::printf("ok\n");
  {  // blocks taken by one thread and given back by others, under memory pressure
    g_capacity = 3000 * KB;
    BlockPool a(false, 256 * KB), b(false, 256 * KB);
    std::atomic<int> bad{0};
    std::vector<std::thread> ts;
    std::mutex qm;
    std::vector<std::pair<BlockPool*, int*>> handed;
    for (int t = 0; t < 6; ++t)
      ts.emplace_back([&, t] {
        unsigned s = 12345u + t;
        for (int i = 0; i < 4000; ++i) {
          s = s * 1664525u + 1013904223u;
          BlockPool* pool = (s >> 20) & 1 ? &a : &b;
          int* p = nullptr;
          if (pool->get(&p, (4 + (s >> 24) % 60) * KB) == hipSuccess) {
            p[0] = t, p[1000] = i;
            std::lock_guard<std::mutex> lock(qm);
            if (p[0] != t || p[1000] != i) ++bad;
            p[0] = -7, p[1000] = -7;
            handed.emplace_back(pool, p);
          }
          std::pair<BlockPool*, int*> g{nullptr, nullptr};
          {
            std::lock_guard<std::mutex> lock(qm);
            if (handed.size() > 20) {
              const size_t k = s % handed.size();
              g = handed[k];
              handed[k] = handed.back();
              handed.pop_back();
            }
          }
          if (g.second) {
            if (g.second[0] != -7 || g.second[1000] != -7) ++bad;  // another owner wrote to it
            g.first->put(g.second);
          }
        }
      });
    for (auto& t : ts) t.join();
    for (auto& g : handed) g.first->put(g.second);
    expect(bad == 0, "one owner at a time");
  }
  expect(g_used == 0, "nothing is left");
  std::printf("ok\n");
}
