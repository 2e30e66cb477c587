// Shared prepass of the fused forward and the adjoint: bounding box, 30-bit
// Morton keys, the stable sort of (key, index) and the packed FP64 record
// gather.  Sets of up to kBlockSortMax particles are sorted by two kernels
// here, larger ones by hipCUB's radix sort.  Kernels live in an anonymous namespace: each translation unit that
// includes this header gets its own copies.
#pragma once

#include <hipcub/hipcub.hpp>

#include "vpm_common.h"

namespace vpm {

namespace {

constexpr int kPreBlock = 256;
constexpr int kBboxBlocks = 512;

__global__ __launch_bounds__(kPreBlock) void bbox_partial_kernel(const double* __restrict__ pos,
                                                                 int64_t ld, int n,
                                                                 double* __restrict__ part) {
  __shared__ double red[6][kPreBlock / 64];
  double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int i = blockIdx.x * kPreBlock + threadIdx.x; i < n; i += gridDim.x * kPreBlock) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double v = pos[c * ld + i];
      mn[c] = fmin(mn[c], v);
      mx[c] = fmax(mx[c], v);
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    mn[c] = wave_min(mn[c]);
    mx[c] = wave_max(mx[c]);
    if (lane == 0) {
      red[c][wave] = mn[c];
      red[3 + c][wave] = mx[c];
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    double v = red[threadIdx.x][0];
    for (int w = 1; w < kPreBlock / 64; ++w)
      v = threadIdx.x < 3 ? fmin(v, red[threadIdx.x][w]) : fmax(v, red[threadIdx.x][w]);
    part[blockIdx.x * 6 + threadIdx.x] = v;
  }
}

// One wave: each lane folds a strided share of the nb partial boxes, then
// the wave reduces (min/max are exact in any order).
__global__ __launch_bounds__(64) void bbox_final_kernel(const double* __restrict__ part, int nb,
                                                        double* __restrict__ bbox) {
  double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int b = threadIdx.x; b < nb; b += 64) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      mn[c] = fmin(mn[c], part[b * 6 + c]);
      mx[c] = fmax(mx[c], part[b * 6 + 3 + c]);
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    mn[c] = wave_min(mn[c]);
    mx[c] = wave_max(mx[c]);
  }
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      bbox[c] = mn[c];
      bbox[3 + c] = mx[c];
    }
  }
}

__device__ inline uint32_t spread10(uint32_t v) {
  v &= 0x3ffu;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

__device__ inline uint32_t morton_key(const double* __restrict__ pos, int64_t ld, int i,
                                      const double* bbox) {
  uint32_t q[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double lo = bbox[c], ext = bbox[3 + c] - lo;
    const double f = ext > 0.0 ? (pos[c * ld + i] - lo) / ext : 0.0;
    int v = static_cast<int>(f * 1023.0);
    v = v < 0 ? 0 : (v > 1023 ? 1023 : v);
    q[c] = static_cast<uint32_t>(v);
  }
  return spread10(q[0]) | (spread10(q[1]) << 1) | (spread10(q[2]) << 2);
}

__global__ __launch_bounds__(kPreBlock) void morton_kernel(const double* __restrict__ pos,
                                                           int64_t ld, int n,
                                                           const double* __restrict__ bbox,
                                                           uint32_t* __restrict__ keys,
                                                           int* __restrict__ idx) {
  const int i = blockIdx.x * kPreBlock + threadIdx.x;
  if (i >= n) return;
  keys[i] = morton_key(pos, ld, i, bbox);
  idx[i] = i;
}

// ---- sort of small sets: sorted blocks, then every particle's rank --------
// A radix sort of some ten thousand keys is a dozen launches of 4-6 us each,
// whatever its size.  Here one kernel sorts blocks of 1024 keys in registers
// and LDS, and a second adds up a key's positions in all blocks, which is its
// place in the whole order (equal keys in index order: the sort is stable).
// Bound by latency: the searches cost n^2 / 1024 binary searches, split over
// eight lanes per key.
constexpr int kSortBlock = 1024;
constexpr int kSamples = 32;     // per block: the last key of each 32
// Velocity of a cloud, radix sort and gather / these kernels: 8,193 particles
// 84 / 66 us, 20,011 240 / 210, 34,914 584 / 563, 65,536 1,872 / 1,863;
// 100,000 4,199 / 4,224, 200,000 16,425 / 16,592.
constexpr int kBlockSortMax = 65536;
constexpr int kSortLanes = 8;    // lanes per key in the second kernel

// Folds the partial boxes, makes the block's keys and sorts them (bitonic, on
// key and place in the block).
__global__ __launch_bounds__(kSortBlock) void sort_block_kernel(
    const double* __restrict__ pos, int64_t ld, int n, const double* __restrict__ part, int nb,
    uint32_t* __restrict__ keys, int* __restrict__ idx, uint32_t* __restrict__ samples) {
  __shared__ double box[6];
  __shared__ uint64_t sh[2][kSortBlock];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (wave < 6) {
    const bool lo = wave < 3;
    double v = lo ? INFINITY : -INFINITY;
    for (int b = lane; b < nb; b += 64) {
      const double x = part[b * 6 + wave];
      v = lo ? fmin(v, x) : fmax(v, x);
    }
    v = lo ? wave_min(v) : wave_max(v);
    if (lane == 0) box[wave] = v;
  }
  __syncthreads();
  const int base = blockIdx.x * kSortBlock;
  uint64_t v = ~uint64_t(0);
  if (base + t < n) v = (static_cast<uint64_t>(morton_key(pos, ld, base + t, box)) << 10) | t;
  int flip = 0;
#pragma unroll
  for (int k = 2; k <= kSortBlock; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      uint64_t o;
      if (j >= 64) {
        sh[flip][t] = v;
        __syncthreads();
        o = sh[flip][t ^ j];
        flip ^= 1;
      } else {
        o = __shfl_xor(static_cast<unsigned long long>(v), j, 64);
      }
      const bool low = ((t & k) == 0) == ((t & j) == 0);
      v = (v < o) == low ? v : o;
    }
  }
  const uint32_t key = static_cast<uint32_t>(v >> 10);  // 2^32 - 1 past n
  if (base + t < n) {
    keys[base + t] = key;
    idx[base + t] = base + static_cast<int>(v & 1023);
  }
  if (t % (kSortBlock / kSamples) == kSortBlock / kSamples - 1)
    samples[blockIdx.x * kSamples + t / (kSortBlock / kSamples)] = key;
}

// Eight lanes per key; they also gather its particle's record, one number each.
__global__ __launch_bounds__(kPreBlock) void sort_rank_kernel(
    const vpm_particles_t p, int n, const uint32_t* __restrict__ keys,
    const int* __restrict__ idx, const uint32_t* __restrict__ samples, int* __restrict__ perm,
    Src8* __restrict__ rec) {
  constexpr int kGroup = kSortBlock / kSamples;
  __shared__ uint32_t smp[(kBlockSortMax / kSortBlock) * (kSamples + 1)];
  const int blocks = (n + kSortBlock - 1) / kSortBlock;
  for (int q = threadIdx.x; q < blocks * kSamples; q += kPreBlock)
    smp[q / kSamples * (kSamples + 1) + q % kSamples] = samples[q];
  __syncthreads();
  const int e = blockIdx.x * (kPreBlock / kSortLanes) + threadIdx.x / kSortLanes;
  const int sub = threadIdx.x % kSortLanes;
  if (e >= n) return;  // with its seven fellows: a key's lanes leave together
  const uint32_t key = keys[e];
  const int own = e / kSortBlock;
  int rank = sub == 0 ? e % kSortBlock : 0;
  for (int b = sub; b < blocks; b += kSortLanes) {
    if (b == own) continue;
    const uint32_t below = key + (b < own);  // earlier blocks' equal keys come first
    const uint32_t* s = smp + b * (kSamples + 1);
    int c = 0;
#pragma unroll
    for (int st = kSamples; st > 0; st >>= 1)
      if (c + st <= kSamples && s[c + st - 1] < below) c += st;
    int at = c * kGroup;
    if (c < kSamples) {  // below the group's last key
      const int len = n - b * kSortBlock;
      const uint32_t* kb = keys + b * kSortBlock;
#pragma unroll
      for (int st = kGroup / 2; st > 0; st >>= 1)
        if (at + st <= len && kb[at + st - 1] < below) at += st;
    }
    rank += at;
  }
#pragma unroll
  for (int off = 1; off < kSortLanes; off <<= 1) rank += __shfl_xor(rank, off, 64);
  const int i = idx[e];
  if (sub == 0) perm[rank] = i;
  if (!rec) return;
  const double v = sub < 3   ? p.pos[sub * p.ld + i]
                   : sub < 6 ? p.str[(sub - 3) * p.ld + i]
                   : sub == 6 ? p.sigma[i]
                   : p.nu     ? p.nu[i]
                              : 0.0;
  reinterpret_cast<double*>(rec + rank)[sub] = v;
}

__global__ __launch_bounds__(kPreBlock) void gather_kernel(const vpm_particles_t p, int n,
                                                           const int* __restrict__ perm,
                                                           Src8* __restrict__ out) {
  const int k = blockIdx.x * kPreBlock + threadIdx.x;
  if (k >= n) return;
  const int i = perm ? perm[k] : k;
  Src8 r;
  r.x = p.pos[i];
  r.y = p.pos[p.ld + i];
  r.z = p.pos[2 * p.ld + i];
  r.ax = p.str[i];
  r.ay = p.str[p.ld + i];
  r.az = p.str[2 * p.ld + i];
  r.s = p.sigma[i];
  r.nu = p.nu ? p.nu[i] : 0.0;
  out[k] = r;
}

__global__ void fill_kernel(double* __restrict__ p, int64_t n, double v) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}


// Sorts particles by Morton key of their position.  Returns the permutation
// (sorted k -> caller index) in `perm` and, if `rec` is not null, the packed
// records in that order.  Scratch: bbox_part (kBboxBlocks*6), bbox (8),
// kin (n, and kSamples more up to kBlockSortMax), kout/iin (n each) and
// cub_bytes of hipCUB storage.
inline int morton_sort(const vpm_particles_t* p, double* bbox_part, double* bbox, uint32_t* kin,
                       uint32_t* kout, int* iin, int* perm, void* cub, size_t cub_bytes, Src8* rec,
                       hipStream_t st) {
  const int64_t n = p->n;
  const int ni = static_cast<int>(n);
  const int nbb = static_cast<int>(std::min<int64_t>(kBboxBlocks, ceil_div(n, kPreBlock)));
  hipLaunchKernelGGL(bbox_partial_kernel, dim3(nbb), dim3(kPreBlock), 0, st, p->pos, p->ld, ni,
                     bbox_part);
  VPM_LAUNCH_CHECK("bbox_partial_kernel");
  if (n <= kBlockSortMax) {
    hipLaunchKernelGGL(sort_block_kernel, dim3(static_cast<unsigned>(ceil_div(n, kSortBlock))),
                       dim3(kSortBlock), 0, st, p->pos, p->ld, ni, bbox_part, nbb, kout, iin, kin);
    VPM_LAUNCH_CHECK("sort_block_kernel");
    hipLaunchKernelGGL(sort_rank_kernel,
                       dim3(static_cast<unsigned>(ceil_div(n, kPreBlock / kSortLanes))),
                       dim3(kPreBlock), 0, st, *p, ni, kout, iin, kin, perm, rec);
    VPM_LAUNCH_CHECK("sort_rank_kernel");
    return VPM_OK;
  }
  hipLaunchKernelGGL(bbox_final_kernel, dim3(1), dim3(64), 0, st, bbox_part, nbb, bbox);
  VPM_LAUNCH_CHECK("bbox_final_kernel");
  const int nb = static_cast<int>(ceil_div(n, kPreBlock));
  hipLaunchKernelGGL(morton_kernel, dim3(nb), dim3(kPreBlock), 0, st, p->pos, p->ld, ni, bbox,
                     kin, iin);
  VPM_LAUNCH_CHECK("morton_kernel");
  size_t cb = cub_bytes;
  VPM_HIP_TRY(hipcub::DeviceRadixSort::SortPairs(cub, cb, kin, kout, iin, perm, ni, 0, 30, st));
  if (rec) {
    hipLaunchKernelGGL(gather_kernel, dim3(nb), dim3(kPreBlock), 0, st, *p, ni,
                       static_cast<const int*>(perm), rec);
    VPM_LAUNCH_CHECK("gather_kernel");
  }
  return VPM_OK;
}

inline int sort_temp_bytes(int64_t n, size_t* bytes) {
  *bytes = 0;
  if (n <= kBlockSortMax) return VPM_OK;
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(
      nullptr, *bytes, static_cast<const uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr),
      static_cast<const int*>(nullptr), static_cast<int*>(nullptr), static_cast<int>(n), 0, 30,
      hipStream_t(0));
  if (e != hipSuccess) {
    set_error("hipcub SortPairs size query failed: %s", hipGetErrorString(e));
    return VPM_ERR_LAUNCH;
  }
  return VPM_OK;
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

}  // namespace

}  // namespace vpm
