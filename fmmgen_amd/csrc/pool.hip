// Device memory of the library's buffers (interface in fmm_common.h).
#include <map>
#include <mutex>
#include <unordered_map>

#include "fmm_common.h"

namespace fmm {

namespace {

struct Block {
  size_t bytes;
  int device;
};

struct Idle {
  void* p;
  unsigned epoch;  // build that gave it back
};

using Map = std::multimap<std::pair<int, size_t>, Idle>;
struct Pool {
  std::mutex mu;
  std::unordered_map<void*, Block> blocks;  // every block handed out or kept
  Map idle;                                 // kept blocks by (device, size)
  size_t idle_bytes = 0;
  unsigned epoch = 0;
};
// Never destroyed: buffers of static trees may be freed after any destructor
// of this file would have run.
Pool& pool() {
  static Pool& p = *new Pool();
  return p;
}
thread_local MemScope* t_scope = nullptr;

// Sizes in steps of an eighth of their power of two (at least 512 bytes), so
// that the slightly different sizes of successive trees meet the same blocks.
size_t size_class(size_t bytes) {
  size_t step = 64;
  while (step * 16 <= bytes) step *= 2;
  return (std::max<size_t>(bytes, 512) + step - 1) / step * step;
}

// The functions below are called with the pool's mutex held.
void drop(Pool& P, Map::iterator it) {
  P.idle_bytes -= it->first.second;
  P.blocks.erase(it->second.p);
  (void)hipFree(it->second.p);
  P.idle.erase(it);
}

void shrink_to(Pool& P, size_t bytes) {  // the oldest go first
  while (P.idle_bytes > bytes) {
    auto old = P.idle.begin();
    for (auto it = P.idle.begin(); it != P.idle.end(); ++it)
      if (P.epoch - it->second.epoch > P.epoch - old->second.epoch) old = it;
    drop(P, old);
  }
}

void keep_idle(Pool& P, void* p) {  // no work on the block is pending
  const Block b = P.blocks[p];
  if (b.bytes > kIdleBytes) {
    P.blocks.erase(p);
    (void)hipFree(p);
    return;
  }
  shrink_to(P, kIdleBytes - b.bytes);
  P.idle.insert({{b.device, b.bytes}, {p, P.epoch}});
  P.idle_bytes += b.bytes;
}

}  // namespace

void* device_alloc(size_t bytes) {
  const size_t want = size_class(bytes);
  if (t_scope)
    if (void* p = t_scope->reuse(want)) return p;
  Pool& P = pool();
  int dev = 0;
  FMM_HIP(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lock(P.mu);
    auto it = P.idle.lower_bound({dev, want});
    if (it != P.idle.end() && it->first.first == dev && it->first.second <= want + want / 4) {
      void* p = it->second.p;
      P.idle_bytes -= it->first.second;
      P.idle.erase(it);
      return p;
    }
  }
  void* p = nullptr;
  size_t got = want;
  hipError_t e = hipMalloc(&p, got);
  if (e == hipErrorOutOfMemory) {  // give back what is kept, then ask for no more than is needed
    (void)hipGetLastError();
    {
      std::lock_guard<std::mutex> lock(P.mu);
      shrink_to(P, 0);
      for (MemScope* s = t_scope; s; s = s->outer) {  // hipFree waits for the work on them
        for (auto& f : s->free) {
          P.blocks.erase(f.second);
          (void)hipFree(f.second);
        }
        s->free.clear();
      }
    }
    e = hipMalloc(&p, got);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      got = std::max<size_t>(bytes, 1);
      e = hipMalloc(&p, got);
    }
  }
  FMM_HIP(e);
  std::lock_guard<std::mutex> lock(P.mu);
  P.blocks[p] = Block{got, dev};
  return p;
}

void device_free(void* p) {
  if (!p) return;
  Pool& P = pool();
  {
    std::lock_guard<std::mutex> lock(P.mu);
    if (t_scope) {
      t_scope->free.insert({P.blocks[p].bytes, p});
      return;
    }
    P.blocks.erase(p);
  }
  (void)hipFree(p);  // waits for the device: nothing is known about pending work
}

size_t trim_memory(size_t keep) {
  Pool& P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  shrink_to(P, keep);
  return P.idle_bytes;
}

MemScope::MemScope(hipStream_t s) : st(s), outer(t_scope) {
  t_scope = this;
  Pool& P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  ++P.epoch;
  for (auto it = P.idle.begin(); it != P.idle.end();) {  // unused for too long
    auto cur = it++;
    if (P.epoch - cur->second.epoch > kIdleBuilds) drop(P, cur);
  }
}

MemScope::~MemScope() {
  t_scope = outer;
  const bool idle = hipStreamSynchronize(st) == hipSuccess;
  Pool& P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  for (auto& f : free) {
    if (idle) {
      keep_idle(P, f.second);
    } else {
      P.blocks.erase(f.second);
      (void)hipFree(f.second);
    }
  }
}

void* MemScope::reuse(size_t want) {
  auto it = free.lower_bound(want);
  if (it == free.end() || it->first > want + want / 4) return nullptr;
  void* p = it->second;
  free.erase(it);
  return p;
}

}  // namespace fmm
