// Processing order of a filter's particles for the cloud-weight kernel.
//
// A wavefront gathers prob for the same cloud point under P particles' poses;
// the closer those poses, the fewer cache lines one gather instruction
// touches and the smaller the set of cells resident caches must hold.  The
// particle arrays themselves stay in index order (the reference's sums run
// over that order, ParticleFilter.cpp:151-193), so only the order in which
// the kernel visits particles changes, and with it nothing but speed: each
// particle's weight is computed by one lane exactly as before.
//
// The order is a counting sort of the particles by a 12-bit key that
// interleaves the leading bits of x, y, z and yaw (each quantised over mean
// +- 2 standard deviations, so the levels stay populated however concentrated
// the set is).  Which coordinate gives the next bit is decided per filter
// (order_levels) by what separates the gathers: a cache line is 32 cells of
// one row along x, so poses apart in y or z are on different lines at once,
// poses apart in x rarely are, and a yaw apart moves a point by its range.
// Each bit goes to the coordinate with the largest remaining deviation in
// weights kSep.  Against one bit each in turn (x, y, z, yaw), the weight
// kernel of cells in floating point measured (1000 x 1000 x 200 map, 20,011
// particles within 0.5 m and 0.15 rad, 7,993 points, tilted) 350 instead of 435
// us, 120 instead of 140 us (8,000 within 1 m, 4,001 points); on the 2000 x 2000 x
// 600 map 520 instead of 640 us (20,000 within 1 m, 10,000 points) and 1,918
// instead of 1,940 us
// (100,000 within 0.1 m, 20,000 points).  Weights of half or twice kSep are
// within 3% of it.  A set spread over several metres (global localisation) has
// no two particles on one line; its key orders by region alone (z, y, x in
// turn: 910 instead of 1,020 us for 60,000 particles over 50 m).
//
// No library calls and no memset, so the sequence can be captured into a HIP
// graph; the batched form sorts many filters at once, one filter per grid row
// (blockIdx.y).  A single filter of at most kOneMax particles is sorted by one
// workgroup in one kernel (order_one_kernel); larger ones and batches by four:
//   moments  64 blocks: partial sums of x, y, z, a and their squares; clears the histogram
//   keys     every block derives the levels from the partial sums; key per
//            particle, histogram per block in LDS, added to the global one
//   scan     one workgroup: exclusive scan of the 4,096 counts
//   scatter  order[offset[key]++] = i (order inside a key is arbitrary)
#include <algorithm>

#include "a3d_math.h"

namespace a3d {
namespace {

constexpr int kBT = 1024;  // threads of the single-workgroup kernels

constexpr int kMB = 64;   // blocks of the moments kernel
constexpr int kKT = 256;  // threads per block of the keys and scatter kernels

// The filter of this block: the launch's one, or row base + blockIdx.y of
// the arrays.
struct OrderJob {
  FilterDev f;
  OrderDev o;
  const FilterDev* fs;
  const OrderDev* os;
  uint32_t base;
};

template <bool MANY>
__device__ inline void job_filter(const OrderJob& j, FilterDev& f, OrderDev& o) {
  if (MANY) {
    f = j.fs[j.base + blockIdx.y];
    o = j.os[j.base + blockIdx.y];
  } else {
    f = j.f;
    o = j.o;
  }
}

// Partial sums of x, y, z, a and their squares (in double) per block, and the
// histogram cleared for the keys kernel.
template <bool MANY>
__global__ __launch_bounds__(kKT) void order_moments_kernel(OrderJob j) {
  FilterDev f;
  OrderDev o;
  job_filter<MANY>(j, f, o);
  __shared__ double red[8][kKT / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t gt = blockIdx.x * kKT + tid, gs = kMB * kKT;
  for (uint32_t k = gt; k < kOrderKeys + 1; k += gs) o.hist[k] = 0u;
  double s1[4] = {0, 0, 0, 0}, s2[4] = {0, 0, 0, 0};
  const float* arr[4] = {f.x, f.y, f.z, f.a};
  for (uint32_t i = gt; i < f.n; i += gs) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float v = arr[k][i];
      const double d = isfinite(v) ? (double)v : 0.0;
      s1[k] += d;
      s2[k] += d * d;
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    for (int d = 32; d >= 1; d >>= 1) {
      s1[k] += __shfl_xor(s1[k], d);
      s2[k] += __shfl_xor(s2[k], d);
    }
    if (lane == 0) {
      red[k][wave] = s1[k];
      red[4 + k][wave] = s2[k];
    }
  }
  __syncthreads();
  if (tid < 8) {
    double a = 0.0;
    for (int w = 0; w < kKT / 64; ++w) a += red[tid][w];
    o.part[blockIdx.x * 8 + tid] = a;
  }
}

// Levels of a filter's keys, per coordinate x, y, z, yaw: lo = mean - 2 sd,
// scale = 1024 / sd (0 when sd is 0), 4,096 levels in all, and which
// coordinate gives each of the key's bits, first bit in the lowest pair.
struct OrderLevels {
  float lo[4], scale[4];
  uint32_t seq;
};

constexpr int kKeyBits = 12;
constexpr float kSep[4] = {1.0f / 16.0f, 1.0f, 4.0f, 4.0f};
constexpr double kRegion = 4.0;  // deviation in x or y (metres) from which a set is ordered by region alone

// Called by one whole wavefront with the sums of all n values and squares
// (s1, s2) in every lane.
__device__ inline void order_levels(const double (&s1)[4], const double (&s2)[4], uint32_t n, OrderLevels* lv) {
  const double inv = 1.0 / (double)(n ? n : 1u);
  float w[4];
  bool region = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double mean = s1[k] * inv;
    const double var = s2[k] * inv - mean * mean;
    const double sd = var > 0.0 ? sqrt(var) : 0.0;
    const bool ok = sd > 0.0 && sd < 1e30;
    if (lane_id() == 0) {
      lv->lo[k] = (float)(mean - 2.0 * sd);
      lv->scale[k] = ok ? (float)(1024.0 / sd) : 0.0f;
    }
    w[k] = ok ? (float)sd * kSep[k] : 0.0f;
    if (k < 2) region |= ok && sd > kRegion;
  }
  uint32_t seq = 0;
#pragma unroll
  for (int b = 0; b < kKeyBits; ++b) {
    uint32_t c = 0;
    float best = w[0];
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      if (w[k] > best) {
        best = w[k];
        c = (uint32_t)k;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (c == (uint32_t)k) w[k] *= 0.5f;
    if (region) c = 2u - (uint32_t)(b % 3);
    seq |= c << (2 * b);
  }
  if (lane_id() == 0) lv->seq = seq;
}

// The levels from the partial sums of the moments kernel (its kMB = 64 blocks,
// one per lane).
__device__ inline void order_levels_of_parts(const FilterDev& f, const OrderDev& o, OrderLevels* lv) {
  static_assert(kMB == 64, "one partial sum per lane");
  double s[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) s[k] = o.part[lane_id() * 8 + k];
#pragma unroll
  for (int k = 0; k < 8; ++k)
    for (int d = 32; d >= 1; d >>= 1) s[k] += __shfl_xor(s[k], d);
  const double s1[4] = {s[0], s[1], s[2], s[3]}, s2[4] = {s[4], s[5], s[6], s[7]};
  order_levels(s1, s2, f.n, lv);
}

__device__ inline uint32_t order_level(float v, float lo, float scale) {
  return (uint32_t)fminf(fmaxf((v - lo) * scale, 0.0f), 4095.0f);  // NaN -> 0
}

__device__ inline uint32_t order_key(float x, float y, float z, float a, const OrderLevels& lv) {
  uint32_t qx = order_level(x, lv.lo[0], lv.scale[0]) << 20, qy = order_level(y, lv.lo[1], lv.scale[1]) << 20;
  uint32_t qz = order_level(z, lv.lo[2], lv.scale[2]) << 20, qa = order_level(a, lv.lo[3], lv.scale[3]) << 20;
  const uint32_t seq = (uint32_t)__builtin_amdgcn_readfirstlane((int)lv.seq);
  uint32_t key = 0;
#pragma unroll
  for (int b = 0; b < kKeyBits; ++b) {  // uniform branches: seq is the filter's
    const uint32_t c = (seq >> (2 * b)) & 3u;
    uint32_t& q = c == 0 ? qx : c == 1 ? qy : c == 2 ? qz : qa;
    key = (key << 1) | (q >> 31);
    q <<= 1;
  }
  return key;
}

// Keys, counted per block in LDS and added to the global histogram once per
// occupied key (few global atomics however concentrated the particles are).
template <bool MANY>
__global__ __launch_bounds__(kKT) void order_keys_kernel(OrderJob j) {
  FilterDev f;
  OrderDev o;
  job_filter<MANY>(j, f, o);
  if (blockIdx.x * kKT >= f.n) return;  // whole block past this filter's end (batched launches)
  __shared__ uint32_t h[kOrderKeys];
  __shared__ OrderLevels lv;
  for (uint32_t k = threadIdx.x; k < kOrderKeys; k += kKT) h[k] = 0u;
  if (threadIdx.x < 64) order_levels_of_parts(f, o, &lv);
  __syncthreads();
  const uint32_t i = blockIdx.x * kKT + threadIdx.x;
  if (i < f.n) {
    const uint32_t key = order_key(f.x[i], f.y[i], f.z[i], f.a[i], lv);
    o.key[i] = key;
    atomicAdd(&h[key], 1u);
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < kOrderKeys; k += kKT)
    if (h[k]) atomicAdd(&o.hist[k], h[k]);
}

template <bool MANY>
__global__ __launch_bounds__(kBT) void order_scan_kernel(OrderJob j) {
  FilterDev f;
  OrderDev o;
  job_filter<MANY>(j, f, o);
  // kOrderKeys / kBT consecutive counts per thread
  __shared__ uint32_t part[kBT];
  constexpr int kPer = kOrderKeys / kBT;
  const int tid = threadIdx.x;
  uint32_t* h = o.hist + (size_t)tid * kPer;
  uint32_t s = 0;
  for (int k = 0; k < kPer; ++k) s += h[k];
  part[tid] = s;
  __syncthreads();
  for (int d = 1; d < kBT; d <<= 1) {  // inclusive scan of the per-thread totals
    const uint32_t v = (tid >= d) ? part[tid - d] : 0u;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  uint32_t run = part[tid] - s;  // exclusive
  for (int k = 0; k < kPer; ++k) {
    const uint32_t c = h[k];
    h[k] = run;
    run += c;
  }
}

// order[offset[key]++] = i: a block reserves one range per occupied key and
// places its particles of that key inside it (in arbitrary order).
template <bool MANY>
__global__ __launch_bounds__(kKT) void order_scatter_kernel(OrderJob j) {
  FilterDev f;
  OrderDev o;
  job_filter<MANY>(j, f, o);
  if (blockIdx.x * kKT >= f.n) return;  // whole block past this filter's end (batched launches)
  __shared__ uint32_t cnt[kOrderKeys];
  for (uint32_t k = threadIdx.x; k < kOrderKeys; k += kKT) cnt[k] = 0u;
  __syncthreads();
  const uint32_t i = blockIdx.x * kKT + threadIdx.x;
  uint32_t key = 0, rank = 0;
  if (i < f.n) {
    key = o.key[i];
    rank = atomicAdd(&cnt[key], 1u);
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < kOrderKeys; k += kKT)
    if (cnt[k]) cnt[k] = atomicAdd(&o.hist[k], cnt[k]);  // now the block's base for key k
  __syncthreads();
  if (i < f.n) o.order[cnt[key] + rank] = i;  // < n: the ranges of key k cover exactly its count
}

// The whole sort by one workgroup, for a single filter of at most kBT * K
// particles: the
// fields stay in registers between the passes, the histogram in LDS, and a
// particle's rank inside its key comes from the LDS add that counts it.  The
// moments are sums in 64 bits, as in the four kernels, of the differences to
// particle 0.  Bound by the latency of its dependent phases: 7 us for 1,000
// particles and 16 us for 5,000, where the four kernels take 20 and 22 us and
// three more launches.  Batches keep the four: a workgroup of 16 wavefronts
// waits for a whole free CU beside the other batches' weight kernels (48
// served sessions in 1.99 ms a round instead of 1.84 ms).
template <int K>
__global__ __launch_bounds__(kBT) void order_one_kernel(FilterDev f, OrderDev o) {
  constexpr int kWaves = kBT / 64, kPer = kOrderKeys / kBT;
  __shared__ uint32_t h[kOrderKeys];
  __shared__ double red[8][kWaves];
  __shared__ OrderLevels lv;
  __shared__ uint32_t tot[kWaves];
  const uint32_t tid = threadIdx.x, n = f.n;
  if (n == 0) return;  // uniform
  const int lane = lane_id(), wave = tid >> 6;
  const float* const arr[4] = {f.x, f.y, f.z, f.a};
  float v[K][4];
#pragma unroll
  for (int u = 0; u < K; ++u) {
    const uint32_t i = min(tid + (uint32_t)u * kBT, n - 1);
#pragma unroll
    for (int k = 0; k < 4; ++k) v[u][k] = arr[k][i];
  }
  float origin[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) origin[k] = arr[k][0];
#pragma unroll
  for (int k = 0; k < kPer; ++k) h[k * kBT + tid] = 0u;
  double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int u = 0; u < K; ++u) {
    if (tid + (uint32_t)u * kBT >= n) break;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float d0 = v[u][k] - origin[k];
      const double d = isfinite(d0) ? (double)d0 : 0.0;
      s[k] += d;
      s[4 + k] += d * d;
    }
  }
  // lanes 8 k .. 8 k + 7 end with the wavefront's sum k: each step halves the sums
  // a lane carries (10 exchanges instead of 48)
  double t;
  {
    double a[4], b[2];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      a[k] = ((lane & 32) ? s[4 + k] : s[k]) + __shfl_xor((lane & 32) ? s[k] : s[4 + k], 32);
#pragma unroll
    for (int k = 0; k < 2; ++k)
      b[k] = ((lane & 16) ? a[2 + k] : a[k]) + __shfl_xor((lane & 16) ? a[k] : a[2 + k], 16);
    t = ((lane & 8) ? b[1] : b[0]) + __shfl_xor((lane & 8) ? b[0] : b[1], 8);
    for (int d = 4; d >= 1; d >>= 1) t += __shfl_xor(t, d);
  }
  if ((lane & 7) == 0) red[lane >> 3][wave] = t;
  __syncthreads();
  if (wave == 0) {
    static_assert(kWaves == 16, "two wavefronts' sums per lane");
    t = red[lane >> 3][lane & 7] + red[lane >> 3][8 + (lane & 7)];
    for (int d = 4; d >= 1; d >>= 1) t += __shfl_xor(t, d);
    double s1[4], s2[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      s1[k] = readlane_d(t, 8 * k);
      s2[k] = readlane_d(t, 8 * (k + 4));
    }
    order_levels(s1, s2, n, &lv);
  }
  __syncthreads();
  uint32_t key[K], rank[K];
#pragma unroll
  for (int u = 0; u < K; ++u) {
    key[u] = order_key(v[u][0] - origin[0], v[u][1] - origin[1], v[u][2] - origin[2], v[u][3] - origin[3], lv);
    rank[u] = tid + (uint32_t)u * kBT < n ? atomicAdd(&h[key[u]], 1u) : 0u;
  }
  __syncthreads();
  uint32_t c[kPer], sum = 0;  // exclusive scan of the counts, kPer consecutive ones per thread
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    c[k] = h[tid * kPer + k];
    sum += c[k];
  }
  uint32_t inc = sum;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t t = __shfl_up(inc, d);
    if (lane >= d) inc += t;
  }
  if (lane == 63) tot[wave] = inc;
  __syncthreads();
  uint32_t run = inc - sum;
  for (int w = 0; w < wave; ++w) run += tot[w];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    h[tid * kPer + k] = run;
    run += c[k];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < K; ++u) {
    const uint32_t i = tid + (uint32_t)u * kBT;
    if (i < n) o.order[h[key[u]] + rank[u]] = i;  // < n: a key's ranks cover exactly its count
  }
}

constexpr uint32_t kOneMax = 8 * kBT;

}  // namespace

void launch_order(const FilterDev& f, const OrderDev& o, hipStream_t s) {
  if (f.n == 0) return;
  const uint32_t blocks = (f.n + kKT - 1) / kKT;
  const OrderJob j{f, o, nullptr, nullptr, 0};
  if (f.n <= kOneMax) {
    if (f.n <= kBT) order_one_kernel<1><<<1, kBT, 0, s>>>(f, o);
    else if (f.n <= 4 * kBT) order_one_kernel<4><<<1, kBT, 0, s>>>(f, o);
    else order_one_kernel<8><<<1, kBT, 0, s>>>(f, o);
    return;
  }
  order_moments_kernel<false><<<kMB, kKT, 0, s>>>(j);
  order_keys_kernel<false><<<blocks, kKT, 0, s>>>(j);
  order_scan_kernel<false><<<1, kBT, 0, s>>>(j);
  order_scatter_kernel<false><<<blocks, kKT, 0, s>>>(j);
}

void launch_order_many(const FilterDev* fs, const OrderDev* os, uint32_t count, uint32_t max_n, hipStream_t s) {
  if (count == 0 || max_n == 0) return;
  const uint32_t blocks = (max_n + kKT - 1) / kKT;
  for (uint32_t base = 0; base < count; base += 65535u) {
    const uint32_t rows = std::min(count - base, 65535u);
    const OrderJob j{FilterDev{}, OrderDev{}, fs, os, base};
    order_moments_kernel<true><<<dim3(kMB, rows), kKT, 0, s>>>(j);
    order_keys_kernel<true><<<dim3(blocks, rows), kKT, 0, s>>>(j);
    order_scan_kernel<true><<<dim3(1, rows), kBT, 0, s>>>(j);
    order_scatter_kernel<true><<<dim3(blocks, rows), kKT, 0, s>>>(j);
  }
}

}  // namespace a3d
