// Buffers for the length of one call: device memory and pinned host memory that
// kernels read and write directly.  hipMalloc, hipFree and pinning cost tens of
// microseconds each, as much as the smallest calls' kernels, so a returned
// buffer is kept for the next call of any thread; a buffer is given back only
// once no stream uses it.  The idle buffers of a kind take at most kIdleMax: one
// more frees those given back longest ago, so a large call's buffers don't keep
// the sizes in use out.  They are all freed when device memory runs out, also
// for what does not come from here (dev_malloc).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "a3d_internal.h"

namespace a3d {
namespace {

constexpr size_t kSmallest = 4096;
constexpr size_t kStep = (size_t)16 << 20;
constexpr size_t kIdleMax[2] = {(size_t)256 << 20, (size_t)64 << 20};  // device, host

struct Pool {
  std::mutex mu;
  std::vector<PoolBuf> idle;
  size_t bytes[2] = {0, 0};
};
// never destroyed: buffers may come back while the process ends
Pool& pool() {
  static Pool* p = new Pool();
  return *p;
}

void release(const PoolBuf& b) {
  if (b.host)
    (void)hipHostFree(b.p);
  else
    (void)hipFree(b.p);
}

// Test knob: A3D_NO_PINNED=1, read once, refuses pinned memory.
bool no_pinned() {
  static const bool no = [] {
    const char* v = std::getenv("A3D_NO_PINNED");
    return v && v[0] == '1';
  }();
  return no;
}

hipError_t fresh(PoolBuf& b) { return b.host ? hipHostMalloc(&b.p, b.bytes, hipHostMallocDefault) : hipMalloc(&b.p, b.bytes); }

// Gives the idle buffers back, after an allocation that failed.
void drain() {
  (void)hipGetLastError();
  std::vector<PoolBuf> drop;
  Pool& P = pool();
  {
    std::lock_guard<std::mutex> lock(P.mu);
    drop.swap(P.idle);
    P.bytes[0] = P.bytes[1] = 0;
  }
  for (const PoolBuf& c : drop) release(c);
}

}  // namespace

bool pool_take(PoolBuf& out, bool host, size_t bytes) {
  if (host && no_pinned()) return false;
  PoolBuf b{};
  b.host = host;
  b.bytes = kSmallest;  // powers of two, then whole steps of kStep
  while (b.bytes < bytes && b.bytes < kStep) b.bytes *= 2;
  if (bytes > kStep) b.bytes = (bytes + kStep - 1) / kStep * kStep;
  if (hipGetDevice(&b.dev) != hipSuccess) return false;
  Pool& P = pool();
  {
    std::lock_guard<std::mutex> lock(P.mu);
    for (size_t i = P.idle.size(); i-- > 0;) {
      const PoolBuf& c = P.idle[i];
      if (c.host == host && c.dev == b.dev && c.bytes == b.bytes) {
        out = c;
        P.bytes[host] -= c.bytes;
        P.idle.erase(P.idle.begin() + (ptrdiff_t)i);
        return true;
      }
    }
  }
  if (fresh(b) != hipSuccess) {
    drain();
    b.p = nullptr;
    if (fresh(b) != hipSuccess) {
      (void)hipGetLastError();  // the caller may go on without: no later check reports this
      return false;
    }
  }
  out = b;
  return true;
}

void pool_give(PoolBuf& b) {
  if (!b.p) return;
  Pool& P = pool();
  std::vector<PoolBuf> drop;
  try {  // destructors come here: no exception leaves
    std::lock_guard<std::mutex> lock(P.mu);
    if (b.bytes <= kIdleMax[b.host]) {
      P.idle.push_back(b);
      P.bytes[b.host] += b.bytes;
      b.p = nullptr;
      for (size_t i = 0; P.bytes[b.host] > kIdleMax[b.host];) {  // ends before the one just added
        if (P.idle[i].host != b.host) {
          ++i;
          continue;
        }
        drop.push_back(P.idle[i]);
        P.bytes[b.host] -= P.idle[i].bytes;
        P.idle.erase(P.idle.begin() + (ptrdiff_t)i);
      }
    }
  } catch (...) {  // no room for the lists: the bound is kept by the next call
  }
  if (b.p) release(b);
  b.p = nullptr;
  for (const PoolBuf& c : drop) release(c);
}

hipError_t dev_malloc_bytes(void** p, size_t bytes) {
  *p = nullptr;
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipSuccess) return e;
  drain();
  *p = nullptr;
  e = hipMalloc(p, bytes);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

}  // namespace a3d
