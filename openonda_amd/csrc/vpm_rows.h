// Driver of the FP64 direct sums: every target against every source, one
// target per lane, the sources through scalar loads.
//
// A workgroup owns one row of 64 targets and splits its sources among its 8
// waves; the waves' sums meet in LDS in wave order.  When the rows alone
// cannot fill the device the sources are also split among workgroups
// (grid.y) and a second kernel adds the splits in order, so every result is
// deterministic.
//
// All lanes of a wave pair with the same source, so the source arrays are
// read through scalar loads and enter the FP64 instructions as scalar
// operands: no LDS staging and no barrier in the sweep.  (A 64-byte FP64
// record broadcast from LDS costs 4 x 8 clocks of LDS return per wave and
// source against about 34 clocks of FP64 issue per CU: LDS would bound it.)
#pragma once

#include <algorithm>

#include "vpm_common.h"

namespace vpm {

namespace {

constexpr int kRow = 64;        // targets per workgroup
constexpr int kRowWaves = 8;    // waves per workgroup
constexpr int kRowBlock = kRow * kRowWaves;
constexpr int kRowGroup = 4;    // sources per group of scalar loads

// 1/sqrt(a) for a > 0: the hardware estimate (relative error e about 2^-24)
// and one third-order step, y (1 + r/2 + 3 r^2/8) with r = 1 - a y^2, whose
// remainder 5 r^3/16 is below 2^-66.  a = inf gives NaN, as the reference's
// inf/inf does.
__device__ __forceinline__ double rsq64(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double r = fma(-a * y, y, 1.0);
  return fma(y * r, fma(0.375, r, 0.5), y);
}
// The same with 1/sqrt(inf) = 0: for sums whose reference weight is 1/pow(A),
// which vanishes at infinite distance (NaN stays NaN through y).
__device__ __forceinline__ double rsq64_inf(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double r = fmin(fma(-a * y, y, 1.0), 1.0);
  return fma(y * r, fma(0.375, r, 0.5), y);
}

// Sources (and, in self evaluations, targets).  q: the second vector field
// (strengths; cotangents in the probe adjoint).  s, nu may be null where the
// operator does not read them.
struct RowArgs {
  int64_t m;            // targets
  int64_t n;            // sources
  const double* tpos;   // [3][tld] target positions
  int64_t tld;
  const double* tq;     // [3][tqld] the targets' own vector field, or null
  int64_t tqld;
  const double* ts;     // [m] the targets' radii, or null
  const double* tnu;    // [m] the targets' viscosities, or null
  const double* pos;    // [3][ld]
  int64_t ld;
  const double* q;      // [3][qld]
  int64_t qld;
  const double* s;      // [n]
  const double* nu;     // [n]
  const Src8* rec;      // self evaluations over records: the particles, else null
  double* out[4];       // vector outputs, [3][ld_out] each; a null one is not stored
  int64_t ld_out;
  double* part;         // split partials [split][component][rows * 64], or null
  double* sums;         // one partial per workgroup (scalar operators)
  int splits;
};

struct RowTarget {
  double x, y, z, ax, ay, az;
  double s, hs;         // radius and half of it
  double nu;
  int64_t i;            // index
};

struct RowSource {
  double x, y, z, ax, ay, az, s, nu;
};

typedef __attribute__((address_space(4))) const double scalar_double_t;

// Scalar-loaded view of the sources.
template <class Op>
struct RowSources {
  static constexpr bool kRecords = false;
  scalar_double_t *x, *y, *z, *ax, *ay, *az, *s, *nu;
  __device__ explicit RowSources(const RowArgs& a) {
    x = (scalar_double_t*)a.pos;
    y = (scalar_double_t*)(a.pos + a.ld);
    z = (scalar_double_t*)(a.pos + 2 * a.ld);
    ax = (scalar_double_t*)a.q;
    ay = (scalar_double_t*)(a.q + a.qld);
    az = (scalar_double_t*)(a.q + 2 * a.qld);
    s = (scalar_double_t*)a.s;
    nu = (scalar_double_t*)a.nu;
  }
  __device__ __forceinline__ RowSource at(int64_t j) const {
    RowSource r{x[j], y[j], z[j], ax[j], ay[j], az[j], 0.0, 0.0};
    if constexpr (Op::kRadius) r.s = s[j];
    if constexpr (Op::kNu) r.nu = nu[j];
    return r;
  }
};

// The same of packed records: one 64-byte line per source where the arrays
// take one of each, which evict one another where the arrays lie a multiple of
// 256 KiB apart (see kRowRecordsMin in vpm_forward_rows.h).
template <class Op>
struct RowRecords {
  static constexpr bool kRecords = true;
  scalar_double_t* r;
  __device__ explicit RowRecords(const RowArgs& a) {
    r = (scalar_double_t*)reinterpret_cast<const double*>(a.rec);
  }
  __device__ __forceinline__ RowSource at(int64_t j) const {
    scalar_double_t* q = r + j * 8;
    RowSource v{q[0], q[1], q[2], q[3], q[4], q[5], 0.0, 0.0};
    if constexpr (Op::kRadius) v.s = q[6];
    if constexpr (Op::kNu) v.nu = q[7];
    return v;
  }
};

// Sources [j, j1) that need a test per pair: pair(k, source) for each k.  Two
// loads in flight: one at a time, every source cost its load's whole latency,
// and the wave with the row's own particles held up its workgroup (FP64
// velocity + stretching of 4,096 particles 36.5 -> 34.4 us, LES step of 4,001
// 140.5 -> 138.7); four spill scalar registers (all outputs but PSE of 2,503
// particles 31.6 us with one, 31.0 with two, 32.0 with four).
template <class Src, class F>
__device__ __forceinline__ void row_few(const Src& src, int64_t j, int64_t j1, F pair) {
  for (; j1 - j >= 2; j += 2) {
    const RowSource s0 = src.at(j), s1 = src.at(j + 1);
    pair(j, s0);
    pair(j + 1, s1);
  }
  if (j < j1) pair(j, src.at(j));
}

template <class Op, class Src>
__device__ __forceinline__ void row_sweep(typename Op::Acc& acc, const RowTarget& t,
                                          const Src& src, int64_t j, int64_t j1) {
  for (; j1 - j >= kRowGroup; j += kRowGroup) {
    RowSource s[kRowGroup];
#pragma unroll
    for (int u = 0; u < kRowGroup; ++u) s[u] = src.at(j + u);
#pragma unroll
    for (int u = 0; u < kRowGroup; ++u) Op::pair(acc, t, s[u]);
  }
  for (; j < j1; ++j) Op::pair(acc, t, src.at(j));
}

// The share of [lo, hi) that part k of `parts` sums, whole groups but for the
// last.
__device__ __forceinline__ void row_share(int64_t lo, int64_t hi, int k, int parts, int64_t* b,
                                          int64_t* e) {
  const int64_t groups = (hi - lo + kRowGroup - 1) / kRowGroup;
  const int64_t per = (groups + parts - 1) / parts * kRowGroup;
  *b = lo + k * per < hi ? lo + k * per : hi;
  *e = hi - *b < per ? hi : *b + per;
}

template <class Op, bool RECORDS = false>
__device__ __forceinline__ RowTarget row_target(const RowArgs& a, int64_t i) {
  RowTarget t{};
  t.i = i;
  t.s = 1.0;
  if constexpr (RECORDS) {
    if (i < a.m) {
      const Src8 r = a.rec[i];
      t = RowTarget{r.x, r.y, r.z, r.ax, r.ay, r.az, r.s, 0.0, r.nu, i};
    }
  } else if (i < a.m) {
    t.x = a.tpos[i];
    t.y = a.tpos[a.tld + i];
    t.z = a.tpos[2 * a.tld + i];
    if constexpr (Op::kTargetData) {
      t.ax = a.tq[i];
      t.ay = a.tq[a.tqld + i];
      t.az = a.tq[2 * a.tqld + i];
      t.s = a.ts[i];
      if constexpr (Op::kNu) t.nu = a.tnu[i];
    }
  }
  t.hs = 0.5 * t.s;
  return t;
}

// Sources [b, e) against one target per lane, the row at row0.
template <class Op, class Src>
__device__ __forceinline__ void row_range(typename Op::Acc& acc, const RowTarget& t,
                                          const Src& src, int64_t row0, int64_t b, int64_t e) {
  if constexpr (Op::kSkipSelf) {  // the row's own particles [o0, o1): j != i
    const int64_t o0 = row0 < b ? b : (row0 < e ? row0 : e);
    const int64_t o1 = row0 + kRow < b ? b : (row0 + kRow < e ? row0 + kRow : e);
    row_few(src, o0, o1, [&](int64_t j, const RowSource& s) {
      if (j != t.i) {
        Op::pair(acc, t, s);
      } else {
        if constexpr (Op::kSelfTerm) Op::self(acc, t);
      }
    });
#pragma unroll 1
    for (int side = 0; side < 2; ++side) row_sweep<Op>(acc, t, src, side ? o1 : b, side ? e : o0);
  } else {
    row_sweep<Op>(acc, t, src, b, e);
  }
}

// Value q of target i: to its split's partials, or to the output.
__device__ __forceinline__ void row_store(const RowArgs& a, int na, int q, int64_t pm, int64_t i,
                                          double s) {
  if (a.part)
    a.part[(static_cast<int64_t>(blockIdx.y) * na + q) * pm + i] = s;
  else if (i < a.m && a.out[q / 3])
    a.out[q / 3][(q % 3) * a.ld_out + i] = s;
}

// Vector operators.  grid (rows, splits).
template <class Op, class Src>
__global__ __launch_bounds__(kRowBlock, 4) void row_kernel(RowArgs a) {
  constexpr int NA = Op::kOut;               // vector components
  constexpr int NV = NA + (Op::kSum ? 1 : 0);  // + one scalar summed over the targets
  __shared__ double red[kRowWaves][NV][kRow];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kRow;
  const RowTarget t = row_target<Op, Src::kRecords>(a, row0 + lane);
  const Src src(a);
  int64_t b, e;
  row_share(0, a.n, static_cast<int>(blockIdx.y) * kRowWaves + wave, a.splits * kRowWaves, &b, &e);
  typename Op::Acc acc{};
  row_range<Op>(acc, t, src, row0, b, e);
  double v[NV];
  Op::result(acc, t, v);
#pragma unroll
  for (int q = 0; q < NV; ++q) red[wave][q][lane] = v[q];
  __syncthreads();
  for (int q = wave; q < NV; q += kRowWaves) {  // one wave per component
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) s += red[w][q][lane];
    const int64_t i = row0 + lane;
    if (q == NA) {
      s = wave_sum(i < a.m ? s : 0.0);
      if (lane == 0) a.sums[static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x] = s;
    } else {
      row_store(a, NA, q, static_cast<int64_t>(gridDim.x) * kRow, i, s);
    }
  }
}

// The same with a row per wave: all eight waves sweep the same sources, held
// together by a barrier per kWideTile, so that a source's cache lines are
// fetched once for 512 targets.  grid (ceil(rows / 8), splits).
constexpr int kWideTile = 512;

template <class Op>
__global__ __launch_bounds__(kRowBlock, 4) void row_wide_kernel(RowArgs a, int rows) {
  constexpr int NA = Op::kOut;
  constexpr int NV = NA + (Op::kSum ? 1 : 0);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = static_cast<int>(blockIdx.x) * kRowWaves + wave;
  const int64_t row0 = static_cast<int64_t>(row) * kRow;
  const RowTarget t = row_target<Op>(a, row0 + lane);
  const RowSources<Op> src(a);
  int64_t b, e;
  row_share(0, a.n, static_cast<int>(blockIdx.y), a.splits, &b, &e);
  typename Op::Acc acc{};
#pragma unroll 1
  for (; b < e; b += kWideTile) {  // the same trips in every wave
    __syncthreads();
    row_range<Op>(acc, t, src, row0, b, e - b < kWideTile ? e : b + kWideTile);
  }
  if (row >= rows) return;
  double v[NV];
  Op::result(acc, t, v);
  const int64_t i = row0 + lane;
#pragma unroll
  for (int q = 0; q < NA; ++q) row_store(a, NA, q, static_cast<int64_t>(rows) * kRow, i, v[q]);
  if constexpr (Op::kSum) {
    const double s = wave_sum(i < a.m ? v[NA] : 0.0);
    if (lane == 0) a.sums[static_cast<int64_t>(blockIdx.y) * rows + row] = s;
  }
}

// When a row per wave pays (sums over arrays; the fused pass has records
// there): the component arrays lie a multiple of 4 MiB apart, so a source's
// seven values fall into the same cache sets, and eight waves at eight places
// of them evict each other's lines.  Velocity of 2^20 particles 1465 -> 1066 ms,
// of 2^19 327 -> 262; stretching of 2^20 2343 -> 1649.  2^18, 2 MiB apart, keeps
// the eight-fold split: 62 ms against 65.  Odd multiples of 2 MiB and less are
// not in the rule, though they collide from 393,216 particles on (786,432: 832
// ms, 579 with a row per wave; 425,984: 217 and 214).  row_splits, made for
// eight waves that share a row's sources, is not tuned for this kernel: these
// sizes have rows enough for one or two splits.
constexpr int64_t kWideStride = int64_t{1} << 19, kWideMin = int64_t{1} << 18;
// The same for up to eight sources at very many points, where eight waves per
// row would have one source each (a million points: velocity of one source 29 ->
// 13 us, of eight about 35 -> 17).
constexpr int64_t kWideSources = 8, kWideRows = 6144;
inline bool row_wide_wanted(const RowArgs& a, int64_t rows) {
  if (a.n <= kWideSources && rows >= kWideRows) return true;
  return a.ld % kWideStride == 0 && a.n >= kWideMin && rows >= kWideMin / kRow;
}

// Adds the splits in order.  grid (targets / 256, components).
__global__ __launch_bounds__(256) void row_reduce_kernel(RowArgs a, int na, int64_t pm) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int q = blockIdx.y;
  if (i >= a.m || !a.out[q / 3]) return;
  double s = 0.0;
  for (int k = 0; k < a.splits; ++k) s += a.part[(static_cast<int64_t>(k) * na + q) * pm + i];
  a.out[q / 3][(q % 3) * a.ld_out + i] = s;
}

// Symmetric scalar sums over pairs i != j (each unordered pair once, counted
// twice) and, with kDiagonal, the pairs i = j.  A workgroup owns rows b and
// R - 1 - b, whose sources j >= row start add up to the same number for every
// b.  grid (ceil(R / 2), splits).
template <class Op>
__global__ __launch_bounds__(kRowBlock, 4) void row_scalar_kernel(RowArgs a, int rows) {
  __shared__ double red[kRowWaves];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const RowSources<Op> src(a);
  double v = 0.0;
#pragma unroll 1
  for (int half = 0; half < 2; ++half) {
    const int row = half ? rows - 1 - static_cast<int>(blockIdx.x) : static_cast<int>(blockIdx.x);
    if (half && row == static_cast<int>(blockIdx.x)) break;
    const int64_t row0 = static_cast<int64_t>(row) * kRow;
    const RowTarget t = row_target<Op>(a, row0 + lane);
    int64_t b, e;
    row_share(row0, a.n, static_cast<int>(blockIdx.y) * kRowWaves + wave, a.splits * kRowWaves, &b,
              &e);
    typename Op::Acc acc{}, own{};
    const int64_t o1 = row0 + kRow < b ? b : (row0 + kRow < e ? row0 + kRow : e);
    for (int64_t j = b; j < o1; ++j) {
      if (j > t.i) Op::pair(acc, t, src.at(j));
      if constexpr (Op::kDiagonal) {
        if (j == t.i) Op::pair(own, t, src.at(j));
      }
    }
    row_sweep<Op>(acc, t, src, o1, e);
    if (t.i < a.m) v += 2.0 * Op::value(acc) + Op::value(own);
  }
  v = block_sum<kRowBlock>(v, red);
  if (threadIdx.x == 0) a.sums[static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x] = v;
}

// Source splits for `groups` workgroups' worth of rows over n sources.  Three
// workgroups fit a CU (768 on the device); equal workgroups run in rounds, a
// round costs a workgroup's sources per wave plus a fixed part (launch,
// target loads, the LDS sum: about 12 sources), and the kernel that adds the
// splits about as much as another 12.  Without splits the 64 rows of 4,096
// points against 131,072 particles would occupy 64 CUs.  Velocity at 1,000 to
// 131,072 particles with 512 or 1024 slots, a fixed part of 6 or 24 or half
// the least share: within 5% either way up to 40,000 and 6% slower at
// 131,072 with other slot counts.
inline int row_splits(int64_t groups, int64_t n) {
  constexpr int64_t kSlots = 768, kFixed = 12;
  if (groups <= 0 || groups >= 8 * kSlots) return 1;
  int best = 1;
  double best_cost = 0.0;
  for (int k = 1; k <= 64; ++k) {
    const double per = static_cast<double>(n) / (static_cast<double>(k) * kRowWaves);
    if (k > 1 && per < 16.0) break;
    const int64_t rounds = (groups * k + kSlots - 1) / kSlots;
    const double cost = static_cast<double>(rounds) * (per + kFixed) + (k > 1 ? kFixed : 0);
    if (k == 1 || cost < best_cost) {
      best = k;
      best_cost = cost;
    }
  }
  return best;
}

inline int64_t row_count(int64_t m) { return ceil_div(m, kRow); }

// Bytes of one split's partials, and of all that row_launch can use for m
// targets and n sources.
inline size_t row_split_bytes(int64_t rows, int na, bool sum) {
  return (static_cast<size_t>(na) * kRow + (sum ? 1 : 0)) * rows * sizeof(double);
}
inline size_t row_workspace_bytes(int64_t m, int64_t n, int na, bool sum = false) {
  const int k = row_splits(row_count(m), n);
  return k > 1 ? k * row_split_bytes(row_count(m), na, sum) : 0;
}

// ws may be null or smaller than row_workspace_bytes: fewer splits then.
// max_splits: 0 or the most splits to use.  kSum operators write one partial
// per workgroup to a.sums (room for the rows), or behind the split partials;
// *sums and *nsums say where and how many.  RECORDS: a.rec may be set.
template <class Op, bool RECORDS = false>
int row_launch(RowArgs a, void* ws, size_t ws_bytes, hipStream_t st, const char* name,
               int max_splits = 0, double** sums = nullptr, int64_t* nsums = nullptr) {
  if (a.m == 0) return VPM_OK;
  const int64_t rows = row_count(a.m);
  const size_t per = row_split_bytes(rows, Op::kOut, Op::kSum);
  int k = row_splits(rows, a.n);
  if (max_splits > 0) k = std::min(k, max_splits);
  if (!ws || ws_bytes / per < 2) k = 1;
  else k = static_cast<int>(std::min<size_t>(k, ws_bytes / per));
  a.splits = k;
  a.part = k > 1 ? static_cast<double*>(ws) : nullptr;
  if constexpr (Op::kSum) {
    if (k > 1) a.sums = a.part + static_cast<int64_t>(k) * Op::kOut * rows * kRow;
    *sums = a.sums;
    *nsums = rows * k;
  }
  const dim3 grid(static_cast<unsigned>(rows), k);
  bool records = false;
  if constexpr (RECORDS) {
    records = a.rec != nullptr;
    if (records)
      hipLaunchKernelGGL((row_kernel<Op, RowRecords<Op>>), grid, dim3(kRowBlock), 0, st, a);
  }
  if (records)
    ;
  else if (row_wide_wanted(a, rows))
    hipLaunchKernelGGL(row_wide_kernel<Op>,
                       dim3(static_cast<unsigned>(ceil_div(rows, kRowWaves)), k), dim3(kRowBlock),
                       0, st, a, static_cast<int>(rows));
  else
    hipLaunchKernelGGL((row_kernel<Op, RowSources<Op>>), grid, dim3(kRowBlock), 0, st, a);
  VPM_LAUNCH_CHECK(name);
  if (k > 1 && Op::kOut > 0) {
    hipLaunchKernelGGL(row_reduce_kernel, dim3(static_cast<unsigned>(ceil_div(a.m, 256)), Op::kOut),
                       dim3(256), 0, st, a, Op::kOut, rows * kRow);
    VPM_LAUNCH_CHECK("row_reduce_kernel");
  }
  return VPM_OK;
}

// Workgroups of row_scalar_kernel for n particles.
inline int64_t row_scalar_blocks(int64_t n, int* splits) {
  const int64_t pairs = (row_count(n) + 1) / 2;
  *splits = row_splits(pairs, n);
  return pairs * *splits;
}

template <class Op>
int row_scalar_launch(RowArgs a, double* sums, int64_t* count, hipStream_t st, const char* name) {
  *count = 0;
  if (a.m == 0) return VPM_OK;
  *count = row_scalar_blocks(a.m, &a.splits);
  a.sums = sums;
  hipLaunchKernelGGL(row_scalar_kernel<Op>, dim3(static_cast<unsigned>(*count / a.splits), a.splits),
                     dim3(kRowBlock), 0, st, a, static_cast<int>(row_count(a.m)));
  VPM_LAUNCH_CHECK(name);
  return VPM_OK;
}

}  // namespace

}  // namespace vpm
