// The device-memory pool (csrc/pool.hip) on a host allocator that stands in for
// the device's: one check a run, named by argv[1]; exit status 0 when it holds.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "fmm_common.h"

namespace {
std::mutex mu;
std::map<void*, size_t> live;
size_t in_use = 0, capacity = ~(size_t)0, mallocs = 0;
thread_local int device = 0;
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lock(mu);
  ++mallocs;
  if (n > capacity || in_use > capacity - n) return hipErrorOutOfMemory;
  static char* next = (char*)0x10000000;  // addresses only: nothing is stored there
  *p = next;
  next += (n + 4095) / 4096 * 4096 + 4096;
  live[*p] = n;
  in_use += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lock(mu);
  auto it = live.find(p);
  if (it == live.end()) {
    std::printf("freed twice or never allocated\n");
    std::abort();
  }
  in_use -= it->second;
  live.erase(it);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }
}

#define CHECK(x)                                         \
  do {                                                   \
    if (!(x)) {                                          \
      std::printf("line %d: %s\n", __LINE__, #x);        \
      return 1;                                          \
    }                                                    \
  } while (0)

using namespace fmm;
constexpr size_t MB = (size_t)1 << 20, GB = (size_t)1 << 30;

static void build(std::vector<size_t> sizes) {  // a build that frees what it allocates
  MemScope scope(nullptr);
  std::vector<void*> v;
  for (size_t s : sizes) v.push_back(device_alloc(s));
  for (void* p : v) device_free(p);
}

// Blocks freed inside a build are given back when a later allocation of the same
// build does not fit beside them.
static int scope_gives_back() {
  capacity = 100 * MB;
  MemScope scope(nullptr);
  for (int k = 0; k < 3; ++k) {
    void* a = device_alloc(60 * MB);
    device_free(a);
    void* b = device_alloc((90 - k) * MB);  // too large for the freed block to serve
    device_free(b);
    void* c = device_alloc(20 * MB);
    device_free(c);
  }
  return 0;
}

// A buffer that fits by its own size, but not by its size class, is still allocated.
static int exact_size() {
  capacity = 1000 * MB;
  void* p = device_alloc(999 * MB);
  CHECK(in_use == 999 * MB);
  {
    MemScope scope(nullptr);
    device_free(p);
    void* q = device_alloc(990 * MB);
    CHECK(in_use <= 1000 * MB);
    device_free(q);
  }
  return 0;
}

// Kept blocks are given back when an allocation fails.
static int idle_gives_back() {
  build({40 * MB, 30 * MB});
  CHECK(in_use >= 70 * MB);
  capacity = 100 * MB;
  void* p = device_alloc(95 * MB);
  CHECK(in_use <= 100 * MB);
  device_free(p);
  return 0;
}

// At most kIdleBytes stay, none longer than kIdleBuilds builds without use, and
// a block is reused by the builds that follow.
static int bounded() {
  for (int k = 0; k < 8; ++k) build({GB + (size_t)k * 300 * MB});
  CHECK(in_use <= kIdleBytes);
  build({kIdleBytes + 1});
  CHECK(in_use <= kIdleBytes);
  build({10 * MB});
  const size_t n = mallocs;
  for (int k = 0; k < 5; ++k) build({10 * MB});
  CHECK(mallocs == n);
  for (unsigned k = 0; k < kIdleBuilds + 2; ++k) build({});
  CHECK(in_use == 0);
  return 0;
}

// Threads with builds of their own, blocks handed from one to the other.
static int threads() {
  std::vector<std::thread> t;
  for (int k = 0; k < 8; ++k)
    t.emplace_back([k] {
      for (int i = 0; i < 2000; ++i) build({(size_t)(1 + (i * 7 + k) % 13) * MB, (size_t)(1 + i % 5) * 1000});
    });
  for (auto& x : t) x.join();
  CHECK(in_use <= kIdleBytes);
  for (unsigned k = 0; k < kIdleBuilds + 2; ++k) build({});
  CHECK(in_use == 0);
  return 0;
}

// On request: all of it, or down to a size.
static int trim() {
  build({40 * MB});
  build({20 * MB, 30 * MB});
  CHECK(trim_memory(60 * MB) <= 60 * MB && in_use <= 60 * MB && in_use >= 50 * MB);  // the oldest went
  void* p = device_alloc(5 * MB);
  CHECK(trim_memory(0) == 0);
  CHECK(in_use >= 5 * MB && in_use < 7 * MB);  // what is in use stays
  device_free(p);
  CHECK(in_use == 0);
  return 0;
}

// A block goes to builds on its own device only.
static int devices() {
  build({50 * MB});
  const size_t n = mallocs;
  device = 1;
  build({50 * MB});
  CHECK(mallocs == n + 1);
  device = 0;
  build({50 * MB});
  CHECK(mallocs == n + 1);
  return 0;
}

// The list buffers of a build: proportional to small sets, a few GiB for the largest.
static int list_buffers() {
  CHECK(list_entries(1) == 1 << 16);
  CHECK(list_entries((size_t)1 << 20) == 16LL << 20);
  CHECK(list_entries((size_t)1 << 24) == 16LL << 24);
  CHECK(8 * list_entries(((size_t)1 << 31) - 1) <= 2LL << 30);
  return 0;
}

int main(int argc, char** argv) {
  const std::map<std::string, int (*)()> checks = {
      {"scope_gives_back", scope_gives_back}, {"exact_size", exact_size}, {"idle_gives_back", idle_gives_back},
      {"bounded", bounded},                   {"threads", threads},       {"devices", devices},
      {"trim", trim},                         {"list_buffers", list_buffers}};
  auto it = argc > 1 ? checks.find(argv[1]) : checks.end();
  if (it == checks.end()) return 2;
  try {
    return it->second();
  } catch (const Error& e) {
    std::printf("%s\n", e.msg.c_str());
    return 3;
  }
}
