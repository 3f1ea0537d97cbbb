// The buffer pool (pool.cpp) over a stand-in for the HIP allocator with a fixed
// capacity: reuse, bounds, eviction, and what happens when memory runs out.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "../../amcl3d_amd/csrc/a3d_internal.h"

namespace {
std::map<void*, size_t> live[2];  // device, host
size_t used[2] = {0, 0}, capacity[2] = {(size_t)4 << 30, (size_t)4 << 30};
long calls = 0;
hipError_t last = hipSuccess;
char* next = nullptr;

hipError_t give(void** p, size_t n, int host) {
  ++calls;
  *p = nullptr;
  if (used[host] + n > capacity[host]) return last = hipErrorOutOfMemory;
  *p = next += 256;
  live[host][*p] = n;
  used[host] += n;
  return hipSuccess;
}
hipError_t take_back(void* p, int host) {
  if (!p) return hipSuccess;
  auto it = live[host].find(p);
  if (it == live[host].end()) {
    std::printf("freed twice, or as the wrong kind\n");
    std::exit(1);
  }
  used[host] -= it->second;
  live[host].erase(it);
  return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return give(p, n, 0); }
hipError_t hipFree(void* p) { return take_back(p, 0); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return give(p, n, 1); }
hipError_t hipHostFree(void* p) { return take_back(p, 1); }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
}

#define CHECK(x)                                            \
  do {                                                      \
    if (!(x)) {                                             \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);   \
      return 1;                                             \
    }                                                       \
  } while (0)

int main() {
  using namespace a3d;
  constexpr size_t kMiB = (size_t)1 << 20;
  const size_t bound[2] = {256 * kMiB, 64 * kMiB};
  for (int host = 0; host < 2; ++host) {
    {  // a returned buffer serves the next call of its size
      Pooled a;
      CHECK(a.take(host, 5000));
    }
    const long before = calls;
    for (int k = 0; k < 10; ++k) {
      Pooled a;
      CHECK(a.take(host, 6000));
    }
    CHECK(calls == before);
    {  // a few large buffers fill the idle bound
      Pooled a, b;
      CHECK(a.take(host, bound[host] / 2));
      CHECK(b.take(host, bound[host] / 2 - 16 * kMiB));
    }
    CHECK(used[host] <= bound[host]);
    for (size_t n : {(size_t)100, (size_t)40000, 3 * kMiB, 20 * kMiB}) {  // other sizes are kept all the same
      { Pooled a; CHECK(a.take(host, n)); }
      const long was = calls;
      for (int k = 0; k < 5; ++k) {
        Pooled a;
        CHECK(a.take(host, n));
      }
      CHECK(calls == was);
      CHECK(used[host] <= bound[host]);
    }
    {  // more than the bound: freed at once, and nothing else goes with it
      const size_t was = used[host];
      { Pooled a; CHECK(a.take(host, bound[host] + 1)); }
      CHECK(used[host] == was);
    }
  }
  // memory runs out: idle buffers are given back, first of all to direct allocations
  CHECK(used[0] > 0);
  capacity[0] = 300 * kMiB;
  void* p = nullptr;
  CHECK(dev_malloc(&p, 290 * kMiB) == hipSuccess);
  CHECK(used[0] == 290 * kMiB);
  float* f = nullptr;
  CHECK(dev_malloc(&f, 20 * kMiB) != hipSuccess && !f);
  CHECK(hipGetLastError() == hipSuccess);  // a later check does not report it
  {
    Pooled a;
    CHECK(!a.take(false, 20 * kMiB) && !a.p);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(a.take(false, 1000));
  }
  CHECK(hipFree(p) == hipSuccess);
  std::printf("ok\n");
  return 0;
}
