// pcl::VoxelGrid<pcl::PointXYZ> on the device, as the node applies it to
// every scan before ParticleFilter::update (Node.cpp:130-141: setLeafSize
// with voxel_size on all three axes, PCL defaults otherwise).
//
// PCL 1.7.2's VoxelGrid::applyFilter, with its defaults (no filter field,
// min_points_per_voxel 0, downsample_all_data true), computes:
//   inv = 1.0f / leaf; min_p, max_p over the finite points;
//   (int64)((max_p - min_p) * inv) + 1 voxels per axis, and if their product
//   exceeds INT32_MAX the input is returned unchanged;
//   min_b = (int)floor(min_p * inv), div_b = floor(max_p * inv) - min_b + 1;
//   per finite point idx = ijk0 + ijk1 * div0 + ijk2 * div0 * div1 with
//   ijk = (int)(floor(p * inv) - (float)min_b), all in float;
//   one output point per distinct idx, in increasing idx, at the float
//   centroid (sum of x, y, z in order, divided by the count as float).
// Here the points of one voxel are summed in point-index order.  PCL's
// std::sort leaves them in an order of its own, so a centroid of three or more
// points can differ from PCL's in the last bits; the voxel set and its order
// are the same.
//
// Lattices of up to kMaxLattice voxels (a 0.1 m leaf over 50 x 50 x 26 m) are
// ranked through a bitmap, one bit per voxel: the number of marked voxels
// below a point's is its output position, and the points are placed in their
// voxel's list without a sort.  Larger ones (and clouds of more than
// kMaxBitmapPoints) radix sort the (idx, point) pairs, which is stable.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cfloat>
#include <vector>

#include "a3d_math.h"

namespace a3d {
namespace {

constexpr int kVT = 1024;
constexpr uint32_t kNoVoxel = 0xffffffffu;

struct VoxelMeta {
  float inv;
  uint32_t nfin;
  int overflow;
  int min_b[3];
  int div[3];
  int mul[3];
};

__device__ inline bool finite3(const float* p) { return isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]); }

__device__ inline const float* point_at(const uint8_t* base, size_t stride, uint32_t i) {
  return reinterpret_cast<const float*>(base + (size_t)i * stride);
}

struct VoxelBounds {
  float lo[3], hi[3];
  uint32_t n;
  uint32_t pad_;
};
constexpr uint32_t kBoundsBlocks = 64;

// Bounds and number of the finite points, per workgroup (one workgroup over all
// of 100,000 points took 66 us, this and the lattice kernel 8 us).
__global__ __launch_bounds__(kVT) void voxel_bounds_kernel(const uint8_t* pts, uint32_t n, size_t stride,
                                                           VoxelBounds* out) {
  __shared__ VoxelBounds red[kVT / 64];
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  VoxelBounds b{{FLT_MAX, FLT_MAX, FLT_MAX}, {-FLT_MAX, -FLT_MAX, -FLT_MAX}, 0u, 0u};
  for (uint32_t i = blockIdx.x * kVT + threadIdx.x; i < n; i += kBoundsBlocks * kVT) {
    const float* p = point_at(pts, stride, i);
    if (!finite3(p)) continue;
    ++b.n;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      b.lo[k] = fminf(b.lo[k], p[k]);
      b.hi[k] = fmaxf(b.hi[k], p[k]);
    }
  }
  auto across = [&]() {
    for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        b.lo[k] = fminf(b.lo[k], __shfl_xor(b.lo[k], d));
        b.hi[k] = fmaxf(b.hi[k], __shfl_xor(b.hi[k], d));
      }
      b.n += __shfl_xor(b.n, d);
    }
  };
  across();
  if (lane == 0) red[wave] = b;
  __syncthreads();
  if (wave != 0) return;
  b = VoxelBounds{{FLT_MAX, FLT_MAX, FLT_MAX}, {-FLT_MAX, -FLT_MAX, -FLT_MAX}, 0u, 0u};
  if (lane < kVT / 64) b = red[lane];
  across();
  if (lane == 0) out[blockIdx.x] = b;
}

// One wavefront: the bounds of all the workgroups, and the voxel lattice.
__global__ __launch_bounds__(64) void voxel_meta_kernel(const VoxelBounds* part, float leaf, VoxelMeta* meta,
                                                        VoxelMeta* host) {
  static_assert(kBoundsBlocks == 64, "one workgroup's bounds per lane");
  VoxelBounds b = part[threadIdx.x];
  for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      b.lo[k] = fminf(b.lo[k], __shfl_xor(b.lo[k], d));
      b.hi[k] = fmaxf(b.hi[k], __shfl_xor(b.hi[k], d));
    }
    b.n += __shfl_xor(b.n, d);
  }
  if (threadIdx.x != 0) return;
  const float* lo = b.lo;
  const float* hi = b.hi;
  VoxelMeta m{};
  m.inv = 1.0f / leaf;
  m.nfin = b.n;
  if (b.n > 0) {
    int64_t d[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) d[k] = (int64_t)((hi[k] - lo[k]) * m.inv) + 1;
    m.overflow = (d[0] * d[1] * d[2] > (int64_t)INT32_MAX) ? 1 : 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      m.min_b[k] = (int)floorf(lo[k] * m.inv);
      m.div[k] = (int)floorf(hi[k] * m.inv) - m.min_b[k] + 1;
    }
    m.mul[0] = 1;
    m.mul[1] = m.div[0];
    m.mul[2] = m.div[0] * m.div[1];
  }
  *meta = m;
  *host = m;
}

__device__ inline uint32_t voxel_key(const VoxelMeta& m, const float* p) {
  int ijk[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) ijk[a] = (int)(floorf(p[a] * m.inv) - (float)m.min_b[a]);
  return (uint32_t)(ijk[0] * m.mul[0] + ijk[1] * m.mul[1] + ijk[2] * m.mul[2]);
}

__global__ void voxel_key_kernel(const uint8_t* pts, uint32_t n, size_t stride, const VoxelMeta* meta,
                                 uint32_t* key, uint32_t* val) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const VoxelMeta m = *meta;
  const float* p = point_at(pts, stride, i);
  uint32_t k = kNoVoxel;
  if (finite3(p)) k = voxel_key(m, p);
  key[i] = k;
  val[i] = i;
}

__global__ void voxel_head_kernel(const uint32_t* key, uint32_t n, uint32_t* head) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  head[i] = (key[i] != kNoVoxel && (i == 0 || key[i] != key[i - 1])) ? 1u : 0u;
}

__global__ void voxel_centroid_kernel(const uint8_t* pts, size_t stride, const uint32_t* key, const uint32_t* val,
                                      const uint32_t* head, const uint32_t* pos, uint32_t n, float* ox, float* oy,
                                      float* oz) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !head[i]) return;
  const uint32_t k = key[i];
  float sx = 0.f, sy = 0.f, sz = 0.f;
  uint32_t j = i;
  for (; j < n && key[j] == k; ++j) {
    const float* p = point_at(pts, stride, val[j]);
    sx += p[0];
    sy += p[1];
    sz += p[2];
  }
  const float c = (float)(j - i);
  const uint32_t o = pos[i];
  ox[o] = sx / c;
  oy[o] = sy / c;
  oz[o] = sz / c;
}

__global__ void voxel_copy_kernel(const uint8_t* pts, size_t stride, uint32_t n, float* ox, float* oy, float* oz) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float* p = point_at(pts, stride, i);
  ox[i] = p[0];
  oy[i] = p[1];
  oz[i] = p[2];
}

// ------------------------------------------------------------ bitmap ranking
constexpr uint32_t kMaxLattice = 1u << 26;  // voxels: a bitmap of 8 MB and as much for its prefix
constexpr uint32_t kRankWords = 1024;       // bitmap words per workgroup of the ranking
constexpr uint32_t kMaxBitmapPoints = 1u << 20;

__global__ void voxel_clear_kernel(uint4* p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = make_uint4(0u, 0u, 0u, 0u);
}

// Every finite point's voxel, and its bit.  Atomics of many points on a few words
// queue up (1.8 ns each: 1,000,000 points in 900 voxels took 1,830 us), so a
// workgroup first joins its points' bits word by word in a hash table in LDS and
// sets each word once (1,085 us for that whole call, where 2,650 went before and
// 2,380 with the sort; a scan of 100,000 points 169 instead of 189 us).
// Workgroups of 256 and 512 points join less (1,252 and 1,236 us).
constexpr uint32_t kMarkThreads = 1024;
__global__ __launch_bounds__(kMarkThreads) void voxel_mark_kernel(const uint8_t* pts, uint32_t n, size_t stride,
                                                                  const VoxelMeta* meta, uint32_t* key,
                                                                  uint32_t* bits) {
  constexpr uint32_t kSlots = 2 * kMarkThreads, kFree = 0xffffffffu;  // half empty: every word finds a slot
  __shared__ uint32_t word[kSlots], mask[kSlots];
  const uint32_t tid = threadIdx.x, i = blockIdx.x * kMarkThreads + tid;
#pragma unroll
  for (uint32_t h = tid; h < kSlots; h += kMarkThreads) {
    word[h] = kFree;
    mask[h] = 0u;
  }
  uint32_t k = kNoVoxel;
  if (i < n) {
    const VoxelMeta m = *meta;
    const float* p = point_at(pts, stride, i);
    if (finite3(p)) k = voxel_key(m, p);
    key[i] = k;
  }
  __syncthreads();
  if (k != kNoVoxel) {
    const uint32_t w = k >> 5;
    uint32_t h = (w * 2654435769u) >> (32 - __builtin_ctz(kSlots));
    for (;;) {
      const uint32_t was = atomicCAS(&word[h], kFree, w);
      if (was == kFree || was == w) break;
      h = (h + 1) & (kSlots - 1);
    }
    atomicOr(&mask[h], 1u << (k & 31));
  }
  __syncthreads();
#pragma unroll
  for (uint32_t h = tid; h < kSlots; h += kMarkThreads)
    if (word[h] != kFree) atomicOr(&bits[word[h]], mask[h]);
}

__device__ inline uint32_t block_sum_u(uint32_t v, uint32_t* red) {
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
  if (lane_id() == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  uint32_t t = 0;
  for (uint32_t w = 0; w < blockDim.x / 64; ++w) t += red[w];
  __syncthreads();
  return t;
}

// Marked voxels per kRankWords words.
__global__ __launch_bounds__(kRankWords) void voxel_count_kernel(const uint32_t* bits, uint32_t words, uint32_t* sums) {
  __shared__ uint32_t red[kRankWords / 64];
  const uint32_t i = blockIdx.x * kRankWords + threadIdx.x;
  const uint32_t t = block_sum_u(i < words ? (uint32_t)__popc(bits[i]) : 0u, red);
  if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

// Marked voxels before each word; the last workgroup leaves their number.
__global__ __launch_bounds__(kRankWords) void voxel_rank_kernel(const uint32_t* bits, uint32_t words,
                                                                const uint32_t* sums, uint32_t* before,
                                                                uint32_t* total, uint32_t* host_total) {
  __shared__ uint32_t red[kRankWords / 64];
  const uint32_t tid = threadIdx.x, i = blockIdx.x * kRankWords + tid;
  const int lane = lane_id(), wave = tid >> 6;
  uint32_t s = 0;
  for (uint32_t b = tid; b < blockIdx.x; b += kRankWords) s += sums[b];
  const uint32_t base = block_sum_u(s, red);
  const uint32_t c = i < words ? (uint32_t)__popc(bits[i]) : 0u;
  uint32_t inc = c;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t v = __shfl_up(inc, d);
    if (lane >= d) inc += v;
  }
  if (lane == 63) red[wave] = inc;
  __syncthreads();
  uint32_t r = base + inc - c;
  for (int w = 0; w < wave; ++w) r += red[w];
  if (i < words) before[i] = r;
  if (blockIdx.x == gridDim.x - 1 && tid == kRankWords - 1) *total = *host_total = r + c;
}

// Every point's output voxel (over its key) and its arrival number there.
__global__ void voxel_tally_kernel(uint32_t* key, uint32_t n, const uint32_t* bits, const uint32_t* before,
                                   uint32_t* count, uint32_t* slot) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t k = key[i];
  if (k == kNoVoxel) return;
  const uint32_t w = k >> 5, o = before[w] + (uint32_t)__popc(bits[w] & ((1u << (k & 31)) - 1u));  // < n
  key[i] = o;
  slot[i] = atomicAdd(&count[o], 1u);
}

// Voxels of up to kSortMax points are summed by half a wavefront or one, larger
// ones by a workgroup each.
constexpr uint32_t kSortMax = 1024;

// Where each voxel's list starts: a workgroup takes one range for its voxels
// (the lists' order does not matter).  The voxels of more than kSortMax points
// are listed in crowd (used[0]: list words taken, used[1]: such voxels).
__global__ __launch_bounds__(kVT) void voxel_alloc_kernel(const uint32_t* count, const uint32_t* total, uint32_t* start,
                                                          uint32_t* used, uint32_t* crowd) {
  __shared__ uint32_t red[kVT / 64];
  __shared__ uint32_t base;
  const uint32_t tid = threadIdx.x, o = blockIdx.x * kVT + tid, nv = *total;
  const int lane = lane_id(), wave = tid >> 6;
  if (blockIdx.x * kVT >= nv) return;  // uniform
  const uint32_t c = o < nv ? count[o] : 0u;
  uint32_t inc = c;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t v = __shfl_up(inc, d);
    if (lane >= d) inc += v;
  }
  if (lane == 63) red[wave] = inc;
  __syncthreads();
  uint32_t r = inc - c;
  for (int w = 0; w < wave; ++w) r += red[w];
  if (tid == kVT - 1) base = atomicAdd(used, r + c);
  __syncthreads();
  if (o < nv) start[o] = base + r;
  if (c > kSortMax) crowd[atomicAdd(used + 1, 1u)] = o;
}

__global__ void voxel_place_kernel(const uint32_t* voxel, uint32_t n, const uint32_t* start, const uint32_t* slot,
                                   uint32_t* list) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t o = voxel[i];
  if (o != kNoVoxel) list[start[o] + slot[i]] = i;  // < n: a voxel's slots cover exactly its count
}

// The centroids of voxels of up to kSortMax points.  Half a wavefront takes a
// voxel of up to 32: it orders them by index (a lane's rank is the number of
// smaller ones) and sums them in that order.  A voxel of more points is taken by
// the whole wavefront, which sorts their indices.
__global__ __launch_bounds__(256) void voxel_average_kernel(const uint8_t* pts, size_t stride, const uint32_t* count,
                                                            const uint32_t* start, const uint32_t* list,
                                                            const uint32_t* total, const uint32_t* used, float* ox,
                                                            float* oy, float* oz, uint32_t* host_crowd) {
  constexpr uint32_t kWaves = 4;
  __shared__ float xyz[kWaves][3][kSortMax];
  const int lane = lane_id(), l = lane & 31, half = lane >> 5;
  const uint32_t wave = threadIdx.x >> 6, nv = *total;
  float(&xs)[3][kSortMax] = xyz[wave];
  if (blockIdx.x == 0 && threadIdx.x == 0) *host_crowd = used[1];
  auto put = [&](uint32_t at, uint32_t i) {
    const float* p = point_at(pts, stride, i);
    xs[0][at] = p[0];
    xs[1][at] = p[1];
    xs[2][at] = p[2];
  };
  auto sum = [&](int axis, uint32_t first, uint32_t c, uint32_t o) {
    float s = 0.f;
#pragma unroll 8
    for (uint32_t j = 0; j < c; ++j) s += xs[axis][first + j];
    float* const out = axis == 0 ? ox : axis == 1 ? oy : oz;
    out[o] = s / (float)c;
  };
  for (uint32_t o2 = (blockIdx.x * kWaves + wave) * 2; o2 < nv; o2 += gridDim.x * kWaves * 2) {  // uniform
    const uint32_t o = o2 + half;
    const uint32_t c = o < nv ? count[o] : 0u;
    const bool few = c <= 32;
    const bool have = few && (uint32_t)l < c;
    const uint32_t i = have ? list[start[o] + l] : 0xffffffffu;
    uint32_t rank = 0;
#pragma unroll
    for (int j = 0; j < 32; ++j) rank += (uint32_t)__shfl((int)i, (lane & 32) + j) < i ? 1u : 0u;
    wave_lds_sync();  // the previous voxels' reads precede these writes
    if (have) put(half * 32 + rank, i);
    wave_lds_sync();
    if (few && l < 3 && o < nv) sum(l, half * 32, c, o);  // lanes 0, 1, 2: x, y, z
    uint64_t crowded = __ballot(!few && l == 0);
    while (crowded) {  // uniform
      const int src = (int)__builtin_ctzll(crowded);
      crowded &= crowded - 1;
      const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)o, src);
      const uint32_t cv = (uint32_t)__builtin_amdgcn_readlane((int)c, src);
      if (cv > kSortMax) continue;
      // bitonic sort of the listed points' indices in LDS
      const uint32_t* const lv = list + start[v];
      uint32_t* const si = reinterpret_cast<uint32_t*>(xs[0]);
      uint32_t np = 64;
      while (np < cv) np <<= 1;
      wave_lds_sync();
#pragma unroll
      for (uint32_t k = 0; k < kSortMax / 64; ++k) {
        const uint32_t j = k * 64 + lane;
        if (k * 64 < np) si[j] = j < cv ? lv[j] : 0xffffffffu;
      }
      for (uint32_t k = 2; k <= np; k <<= 1) {
        for (uint32_t d = k >> 1; d > 0; d >>= 1) {
          wave_lds_sync();
          for (uint32_t t = lane; t < np / 2; t += 64) {
            const uint32_t p = 2 * t - (t & (d - 1)), q = p + d;
            const uint32_t x = si[p], y = si[q];
            if ((x > y) == ((p & k) == 0)) {
              si[p] = y;
              si[q] = x;
            }
          }
        }
      }
      wave_lds_sync();
      uint32_t at[kSortMax / 64];
#pragma unroll
      for (uint32_t k = 0; k < kSortMax / 64; ++k) at[k] = k * 64 + lane < cv ? si[k * 64 + lane] : 0u;
      wave_lds_sync();  // the indices have been read: the points go over them
#pragma unroll
      for (uint32_t k = 0; k < kSortMax / 64; ++k)
        if (k * 64 + lane < cv) put(k * 64 + lane, at[k]);
      wave_lds_sync();
      if (lane < 3) sum(lane, 0, cv, v);
    }
  }
}

// The centroids of the voxels in crowd, a workgroup each.  A voxel's points are
// marked in a bitmap over the cloud's indices, kWindow of them at a time; its set
// bits in order are the points in index order, gathered to LDS kVT at a time and
// summed in that order.  Bound by the adds (three lanes, one dependent add per
// point).  A wavefront that searched all the cloud's points for each such voxel
// took 2.2 ms (900 voxels of 1,100 in 1,000,000 points); this takes 90 us.
constexpr uint32_t kWindow = 1u << 18;
__global__ __launch_bounds__(kVT) void voxel_crowded_kernel(const uint8_t* pts, uint32_t n, size_t stride,
                                                            const uint32_t* count, const uint32_t* start,
                                                            const uint32_t* list, const uint32_t* crowd, float* ox,
                                                            float* oy, float* oz) {
  constexpr uint32_t kPer = kWindow / 32 / kVT;  // bitmap words per thread
  __shared__ uint32_t bits[kWindow / 32];
  __shared__ uint32_t idx[kVT];
  __shared__ float xyz[3][kVT];
  __shared__ uint32_t red[kVT / 64];
  const uint32_t tid = threadIdx.x, v = crowd[blockIdx.x], c = count[v];
  const int lane = lane_id(), wave = tid >> 6;
  const uint32_t* const lv = list + start[v];
  float s = 0.f;  // threads 0, 1, 2: x, y, z
  for (uint32_t w0 = 0; w0 < n; w0 += kWindow) {  // n <= kMaxBitmapPoints: no overflow
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) bits[k * kVT + tid] = 0u;
    __syncthreads();
    for (uint32_t j = tid; j < c; j += kVT) {
      const uint32_t i = lv[j] - w0;  // wraps below the window
      if (i < kWindow) atomicOr(&bits[i >> 5], 1u << (i & 31));
    }
    __syncthreads();
    uint32_t w[kPer], own = 0;  // consecutive words
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
      w[k] = bits[tid * kPer + k];
      own += (uint32_t)__popc(w[k]);
    }
    uint32_t inc = own;
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t t = __shfl_up(inc, d);
      if (lane >= d) inc += t;
    }
    if (lane == 63) red[wave] = inc;
    __syncthreads();
    uint32_t first = inc - own, cw = 0;  // this thread's first point's position, points in the window
    for (uint32_t k = 0; k < kVT / 64; ++k) {
      if (k < (uint32_t)wave) first += red[k];
      cw += red[k];
    }
    for (uint32_t t0 = 0; t0 < cw; t0 += kVT) {  // uniform
      uint32_t q = first;
#pragma unroll
      for (uint32_t k = 0; k < kPer; ++k) {
        uint32_t m = w[k];
        const uint32_t after = q + (uint32_t)__popc(m);
        if (after > t0 && q < t0 + kVT) {
          for (; m; m &= m - 1, ++q)
            if (q - t0 < kVT) idx[q - t0] = w0 + (tid * kPer + k) * 32 + (uint32_t)__builtin_ctz(m);
        }
        q = after;
      }
      __syncthreads();
      const uint32_t len = min((uint32_t)kVT, cw - t0);
      if (tid < len) {
        const float* p = point_at(pts, stride, idx[tid]);
        xyz[0][tid] = p[0];
        xyz[1][tid] = p[1];
        xyz[2][tid] = p[2];
      }
      __syncthreads();
      if (tid < 3) {
#pragma unroll 8
        for (uint32_t j = 0; j < len; ++j) s += xyz[tid][j];
      }
      // idx is written next, xyz only after another barrier
    }
    __syncthreads();  // red and bits have been read
  }
  if (tid < 3) (tid == 0 ? ox : tid == 1 ? oy : oz)[v] = s / (float)c;
}

}  // namespace

// Buffers of voxel_grid_device, kept by a caller that filters many clouds: the
// meta record (with the workgroups' bounds and the voxel count after it), the
// host's copy of the record and the count, the words of the path taken (bitmap
// ranking, or the sort's keys, values, their sorted copies, voxel heads and
// positions) and the sort / scan temporary.
struct VoxelWorkspace {
  Pooled meta, host, buf, tmp;
};

VoxelWorkspace* voxel_workspace_new() { return new VoxelWorkspace(); }

void voxel_workspace_free(VoxelWorkspace* w) { delete w; }

// d_pts: n points, `stride` bytes apart (x, y, z the first three floats).
// Writes the filtered cloud as d_x, d_y, d_z (capacity n) and its size.
// ws: buffers to reuse (grown as needed), or null for buffers of this call.
int voxel_grid_device(const void* d_pts, size_t n, size_t stride, float leaf, float* d_x, float* d_y, float* d_z,
                      size_t* out_n, hipStream_t s, VoxelWorkspace* ws) {
  *out_n = 0;
  if (n == 0) return A3D_OK;
  const uint8_t* pts = static_cast<const uint8_t*>(d_pts);
  const uint32_t nn = (uint32_t)n;
  const uint32_t blocks = (nn + 255) / 256;
  VoxelWorkspace local;
  VoxelWorkspace& w = ws ? *ws : local;
  uint32_t *key = nullptr, *val = nullptr, *key2 = nullptr, *val2 = nullptr, *head = nullptr, *pos = nullptr;
  size_t tmp_bytes = 0, tmp2 = 0;
  // Every return leaves the stream idle: a buffer that goes back to the pool
  // is not in use.
#define A3D_TRY(call)               \
  if (!hip_ok((call), #call)) {     \
    (void)hipStreamSynchronize(s);  \
    return A3D_ERR_HIP;             \
  }
  // grown only while the stream is idle
  auto grow = [](Pooled& b, bool host, size_t bytes) {
    if (b.p && b.bytes >= bytes) return hipSuccess;
    pool_give(b);
    return b.take(host, bytes) ? hipSuccess : hipErrorOutOfMemory;
  };
  struct Host {
    VoxelMeta meta;
    uint32_t total, crowd;
  };
  constexpr size_t kPartAt = (sizeof(VoxelMeta) + 63) & ~(size_t)63;
  constexpr size_t kTotalAt = kPartAt + kBoundsBlocks * sizeof(VoxelBounds);
  constexpr size_t kHostAt = kTotalAt + 64;
  A3D_TRY(grow(w.meta, false, kHostAt + sizeof(Host)));
  uint8_t* const rec = static_cast<uint8_t*>(w.meta.p);
  VoxelMeta* const meta = reinterpret_cast<VoxelMeta*>(rec);
  VoxelBounds* const part = reinterpret_cast<VoxelBounds*>(rec + kPartAt);
  uint32_t* const total = reinterpret_cast<uint32_t*>(rec + kTotalAt);
  // the kernels write the host's record to pinned memory, or, where there is
  // none, beside the rest, and it is copied
  const bool pinned = grow(w.host, true, sizeof(Host)) == hipSuccess;
  Host copy{};
  Host* const out = pinned ? static_cast<Host*>(w.host.p) : reinterpret_cast<Host*>(rec + kHostAt);
  const Host* const host = pinned ? out : &copy;
  auto wait = [&]() {
    const hipError_t e = pinned ? hipSuccess : hipMemcpyAsync(&copy, out, sizeof(Host), hipMemcpyDeviceToHost, s);
    const hipError_t done = hipStreamSynchronize(s);
    return e != hipSuccess ? e : done;
  };
  voxel_bounds_kernel<<<kBoundsBlocks, kVT, 0, s>>>(pts, nn, stride, part);
  voxel_meta_kernel<<<1, 64, 0, s>>>(part, leaf, meta, &out->meta);
  A3D_TRY(hipGetLastError());
  A3D_TRY(wait());
  const VoxelMeta hm = host->meta;
  if (hm.nfin == 0) return A3D_OK;
  if (hm.overflow) {  // PCL: integer indices would overflow, output = input
    voxel_copy_kernel<<<blocks, 256, 0, s>>>(pts, stride, nn, d_x, d_y, d_z);
    A3D_TRY(hipGetLastError());
    A3D_TRY(hipStreamSynchronize(s));
    *out_n = n;
    return A3D_OK;
  }
  // The bitmap serves a lattice of at most kMaxLattice voxels whose cells are
  // exact floats (a key is then below the lattice's size); clearing and ranking
  // a bitmap much larger than the cloud would cost more than the sort (7.5M
  // voxels take 5 us, 67M 20 us, the sort's extra launches 60 us).
  const double lattice = (double)hm.div[0] * hm.div[1] * hm.div[2];
  bool bitmap = lattice <= (double)kMaxLattice && nn <= kMaxBitmapPoints;
  for (int k = 0; k < 3; ++k)
    bitmap = bitmap && hm.div[k] > 0 && hm.div[k] < (1 << 24) && hm.min_b[k] > -(1 << 30) && hm.min_b[k] < (1 << 30);
  if (bitmap) {
    const uint32_t words = (uint32_t)(((uint64_t)lattice + 31) / 32), wp = (words + 3) & ~3u, np = (nn + 3) & ~3u;
    const uint32_t rank_blocks = (words + kRankWords - 1) / kRankWords;
    A3D_TRY(grow(w.buf, false, (2 * (size_t)wp + 5 * (size_t)np + 4 + rank_blocks + nn / kSortMax) * 4));
    uint32_t* const bits = static_cast<uint32_t*>(w.buf.p);  // cleared together with used and count
    uint32_t* const used = bits + wp;
    uint32_t* const count = used + 4;
    uint32_t* const before = count + np;
    uint32_t* const voxel = before + wp;  // each point's key, then its output voxel
    uint32_t* const slot = voxel + np;
    uint32_t* const start = slot + np;
    uint32_t* const list = start + np;
    uint32_t* const sums = list + np;
    uint32_t* const crowd = sums + rank_blocks;  // fewer than nn / kSortMax voxels hold more than kSortMax
    const uint32_t clear = (wp + 4 + np) / 4;
    voxel_clear_kernel<<<(clear + 255) / 256, 256, 0, s>>>(reinterpret_cast<uint4*>(bits), clear);
    voxel_mark_kernel<<<(nn + kMarkThreads - 1) / kMarkThreads, kMarkThreads, 0, s>>>(pts, nn, stride, meta, voxel, bits);
    voxel_count_kernel<<<rank_blocks, kRankWords, 0, s>>>(bits, words, sums);
    voxel_rank_kernel<<<rank_blocks, kRankWords, 0, s>>>(bits, words, sums, before, total, &out->total);
    voxel_tally_kernel<<<blocks, 256, 0, s>>>(voxel, nn, bits, before, count, slot);
    voxel_alloc_kernel<<<(nn + kVT - 1) / kVT, kVT, 0, s>>>(count, total, start, used, crowd);
    voxel_place_kernel<<<blocks, 256, 0, s>>>(voxel, nn, start, slot, list);
    voxel_average_kernel<<<std::min(1024u, (nn + 7) / 8), 256, 0, s>>>(pts, stride, count, start, list, total, used,
                                                                       d_x, d_y, d_z, &out->crowd);
    A3D_TRY(hipGetLastError());
    A3D_TRY(wait());
    if (host->crowd) {
      voxel_crowded_kernel<<<host->crowd, kVT, 0, s>>>(pts, nn, stride, count, start, list, crowd, d_x, d_y, d_z);
      A3D_TRY(hipGetLastError());
      A3D_TRY(hipStreamSynchronize(s));
    }
    *out_n = host->total;
    return A3D_OK;
  }
  A3D_TRY(grow(w.buf, false, 6 * n * 4));
  key = static_cast<uint32_t*>(w.buf.p);
  val = key + n;
  key2 = val + n;
  val2 = key2 + n;
  head = val2 + n;
  pos = head + n;
  voxel_key_kernel<<<blocks, 256, 0, s>>>(pts, nn, stride, meta, key, val);
  A3D_TRY(hipGetLastError());
  A3D_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, key, key2, val, val2, (int)nn, 0, 32, s));
  A3D_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp2, head, pos, (int)nn, s));
  tmp_bytes = std::max(tmp_bytes, tmp2);
  A3D_TRY(grow(w.tmp, false, std::max(tmp_bytes, (size_t)1)));
  void* const tmp = w.tmp.p;
  A3D_TRY(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, key, key2, val, val2, (int)nn, 0, 32, s));
  voxel_head_kernel<<<blocks, 256, 0, s>>>(key2, nn, head);
  A3D_TRY(hipGetLastError());
  A3D_TRY(hipcub::DeviceScan::ExclusiveSum(tmp, tmp_bytes, head, pos, (int)nn, s));
  voxel_centroid_kernel<<<blocks, 256, 0, s>>>(pts, stride, key2, val2, head, pos, nn, d_x, d_y, d_z);
  A3D_TRY(hipGetLastError());
  uint32_t last[2] = {0, 0};
  A3D_TRY(hipMemcpyAsync(&last[0], pos + (nn - 1), 4, hipMemcpyDeviceToHost, s));
  A3D_TRY(hipMemcpyAsync(&last[1], head + (nn - 1), 4, hipMemcpyDeviceToHost, s));
  A3D_TRY(hipStreamSynchronize(s));
#undef A3D_TRY
  *out_n = (size_t)last[0] + last[1];
  return A3D_OK;
}

}  // namespace a3d
