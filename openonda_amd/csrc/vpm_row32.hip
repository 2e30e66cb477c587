// FP32-compensated pair sums over rows of 64 sorted targets.
//
// A workgroup owns one row; its eight waves take the source chunks in turn
// (chunk c goes to part c mod parts, over the waves and the source splits), so
// a row's few near chunks spread over the waves.  Every lane of a wave pairs
// with the same source, so the sources come through scalar loads from FP32
// records relative to their chunk's centre, and enter the pair instructions
// as scalar operands: no LDS staging, no barrier in the sweep.  (The staged
// form read 48 bytes per source and wave from LDS with per-particle radii,
// 3 x 8 clocks of the CU's LDS return path against about 18 clocks of FP32
// issue: LDS bound it.)  The target's offset to the chunk centre comes from
// FP64 positions once per chunk; FP32 partials of a chunk are folded into
// FP64 totals.
//
// Stretching: waves of coherent strengths (coherent_wave) take the sum of
// g alpha_j and the triple product in FP64 on chunks near the row and in FP32
// on far ones (gap between the boxes above kFarGap32 times the larger
// radius), the others in FP32 everywhere, as in the tiled kernels
// (vpm_fused.hip, which also measures why); sets with vorticity or enstrophy
// and without PSE sum in FP64 on near chunks in every wave.
//
// With s = sigma_ij, D = r^2 + s^2, t = D^-1/2 and w = s^2 t^2 no reciprocal
// of s is needed: (rho^2 + 2.5) / (A^5/2 s^3) = t^3 (1 + 1.5 w) and so on
// (vpm_plain.hip).
//
// Bound: FP32 issue (velocity alone 2.45e12 pairs/s, 1.55 wave64 instructions
// per clock and CU).  Tiled kernels -> here, per call at N = 100,000: velocity
// 4.80 -> 4.17 ms, with per-particle radii 6.80 -> 4.78; stretching of a ring
// 9.51 -> 7.40, 11.5 -> 7.31; PSE 5.81 -> 4.92, 6.96 -> 5.78; vorticity +
// enstrophy 4.97 -> 4.73, 7.41 -> 5.98; all five with per-particle radii 16.0
// -> 14.7 (cloud), 19.4 -> 15.4 (ring); at 8,192 to 35,000 alike.

#include "vpm_row32.h"

#include <algorithm>

#include "vpm_rows.h"

namespace vpm {

namespace {

constexpr int kChunk32 = 64;      // sources per chunk
constexpr int kStride32 = 12;     // most floats per record
constexpr int kGroup32 = 4;       // records per group of scalar loads
constexpr int kBox32 = 8;         // doubles per chunk box: centre, half-extent, largest radius
constexpr double kFarGap32 = 4.0;

// Record layout: offset (3), strength (3), with per-particle radii sigma/2
// and sigma^2, with PSE the low parts alpha - fp32(alpha); lengths in units
// of the first particle's radius.
template <unsigned OUT, bool UNIF>
struct Rec32 {
  static constexpr bool kLo = OUT & VPM_OUT_PSE;
  static constexpr int kLoAt = UNIF ? 6 : 8;
  static constexpr int kStride = kLo ? 12 : (UNIF ? 6 : 8);
};

__device__ __forceinline__ double held(double v) {  // rounded here, not fused into its use
  asm volatile("" : "+v"(v));
  return v;
}

// One workgroup of 64 lanes per chunk.  Lanes past n write zero-strength
// padding far away, which adds exactly 0.
__global__ __launch_bounds__(kChunk32) void row32_records_kernel(const Src8* __restrict__ src,
                                                                 int n, int stride, int lo_at,
                                                                 int unif,
                                                                 float* __restrict__ rec,
                                                                 double* __restrict__ box) {
  const int c = blockIdx.x;
  const int k = c * kChunk32 + static_cast<int>(threadIdx.x);
  const bool ok = k < n;
  const double scale = 1.0 / src[0].s;
  Src8 g{};
  if (ok) g = src[k];
  const double p[3] = {held(g.x * scale), held(g.y * scale), held(g.z * scale)};
  double cen[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const double lo = wave_min(ok ? p[q] : INFINITY), hi = wave_max(ok ? p[q] : -INFINITY);
    cen[q] = 0.5 * (lo + hi);
    if (threadIdx.x == 0) {
      box[static_cast<int64_t>(c) * kBox32 + q] = cen[q];
      box[static_cast<int64_t>(c) * kBox32 + 3 + q] = 0.5 * (hi - lo);
    }
  }
  const double sig = g.s * scale, smax = wave_max(ok ? sig : 0.0);
  if (threadIdx.x == 0) box[static_cast<int64_t>(c) * kBox32 + 6] = smax;
  float* r = rec + static_cast<int64_t>(k) * stride;
  const float ax = static_cast<float>(g.ax), ay = static_cast<float>(g.ay),
              az = static_cast<float>(g.az);
  for (int q = 0; q < 3; ++q) r[q] = ok ? static_cast<float>(p[q] - cen[q]) : 1e18f;
  r[3] = ax;
  r[4] = ay;
  r[5] = az;
  if (!unif) {
    r[6] = ok ? static_cast<float>(0.5 * sig) : 0.5f;
    r[7] = ok ? static_cast<float>(sig * sig) : 1.0f;
  }
  if (stride == 12) {
    r[lo_at] = static_cast<float>(g.ax - static_cast<double>(ax));
    r[lo_at + 1] = static_cast<float>(g.ay - static_cast<double>(ay));
    r[lo_at + 2] = static_cast<float>(g.az - static_cast<double>(az));
    for (int q = lo_at + 3; q < stride; ++q) r[q] = 0.0f;
    for (int q = unif ? 6 : 8; q < lo_at; ++q) r[q] = 0.0f;
  }
}

struct Tgt32 {
  float x, y, z, ax, ay, az, hs, lx, ly, lz;
};

// One pair.  G64: g alpha_j into g64 and the triple product in FP64 from the
// FP64 strengths aj (source) and ai (target).  self: the pair is the target's
// own (its g alpha_i leaves G; every other term but the enstrophy's is 0).
template <unsigned OUT, bool UNIF, bool G64>
__device__ __forceinline__ void pair32(float* acc, double* g64, const Tgt32& t, const float* f,
                                       const double* aj, const double* ai, float eps,
                                       const PairConst<float>& k, bool self) {
  using S = Slots<OUT>;
  const float dx = t.x - f[0], dy = t.y - f[1], dz = t.z - f[2];
  float s = 1.0f, s2 = 1.0f, r2 = 0.0f, D;
  if constexpr (!UNIF) {
    s = t.hs + f[6];
    s2 = s * s;
  }
  if constexpr (S::vort) {
    r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
    D = r2 + s2;
  } else {
    D = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, s2)));
  }
  const float t1 = __builtin_amdgcn_rsqf(D);
  const float t2 = t1 * t1;
  const float t3 = t2 * t1;
  const float w = UNIF ? t2 : s2 * t2;
  if constexpr (S::vel || S::str) {
    const float g = t3 * __builtin_fmaf(k.c15, w, 1.0f);
    const float cx = dy * f[5] - dz * f[4];
    const float cy = dz * f[3] - dx * f[5];
    const float cz = dx * f[4] - dy * f[3];
    if constexpr (S::vel) {
      acc[kU + 0] += g * cx;
      acc[kU + 1] += g * cy;
      acc[kU + 2] += g * cz;
    }
    if constexpr (S::str) {
      const float gG = self ? 0.0f : g;
      float e;
      if constexpr (G64) {
        const double gd = gG;
        g64[0] = fma(gd, aj[0], g64[0]);
        g64[1] = fma(gd, aj[1], g64[1]);
        g64[2] = fma(gd, aj[2], g64[2]);
        const double rx = dx, ry = dy, rz = dz;
        const double qx = ry * aj[2] - rz * aj[1];
        const double qy = rz * aj[0] - rx * aj[2];
        const double qz = rx * aj[1] - ry * aj[0];
        e = static_cast<float>(ai[0] * qx + ai[1] * qy + ai[2] * qz);
      } else {
        acc[kG + 0] += gG * f[3];
        acc[kG + 1] += gG * f[4];
        acc[kG + 2] += gG * f[5];
        e = t.ax * cx + t.ay * cy + t.az * cz;
      }
      const float v = (t3 * t2) * __builtin_fmaf(k.c75, w, k.c3) * e;
      acc[kSd + 0] += v * dx;
      acc[kSd + 1] += v * dy;
      acc[kSd + 2] += v * dz;
    }
  }
  if constexpr (S::pse) {
    const float* lo = f + Rec32<OUT, UNIF>::kLoAt;
    const float v = UNIF ? (t3 * t3) * t3 : (s * t3) * (w * w * w);
    acc[kP + 0] += v * ((f[3] - t.ax) + (lo[0] - t.lx));
    acc[kP + 1] += v * ((f[4] - t.ay) + (lo[1] - t.ly));
    acc[kP + 2] += v * ((f[5] - t.az) + (lo[2] - t.lz));
  }
  if constexpr (S::vort) {
    float v;
    if constexpr (UNIF) {
      v = t3 * (t2 * t2);
    } else {  // sigma_j, not sigma_ij (ParticlesPhysicsCuda.py:323,334-337)
      const float q1 = __builtin_amdgcn_rsqf(r2 + f[7]);
      const float q2 = q1 * q1, wj = f[7] * q2;
      v = (q2 * q1) * (wj * wj);
    }
    v = r2 > eps ? v : 0.0f;
    acc[kW + 0] += v * f[3];
    acc[kW + 1] += v * f[4];
    acc[kW + 2] += v * f[5];
  }
  if constexpr (S::ens) {
    const float v = t1 * __builtin_fmaf(k.c22, w, 1.0f);
    acc[kE + 0] += v * f[3];
    acc[kE + 1] += v * f[4];
    acc[kE + 2] += v * f[5];
  }
}

// grid (rows, splits)
template <unsigned OUT, bool UNIF>
__global__ __launch_bounds__(kRowBlock, 4) void row32_kernel(FusedArgs a, int splits,
                                                             const float* __restrict__ rec_,
                                                             const double* __restrict__ box_) {
  using S = Slots<OUT>;
  using R = Rec32<OUT, UNIF>;
  constexpr int NS = S::nslot;
  __shared__ double red[kRowWaves][NS][kRow];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = blockIdx.x;
  const int kt = row * kRow + lane;
  const bool valid = kt < a.n;
  const double scale = 1.0 / a.src[0].s;
  Src8 ti{0, 0, 0, 0, 0, 0, 1, 0};
  if (valid) ti = a.src[kt];
  const double X = held(ti.x * scale), Y = held(ti.y * scale), Z = held(ti.z * scale);
  Tgt32 t;
  t.ax = static_cast<float>(ti.ax);
  t.ay = static_cast<float>(ti.ay);
  t.az = static_cast<float>(ti.az);
  t.hs = static_cast<float>(0.5 * ti.s * scale);
  t.lx = static_cast<float>(ti.ax - static_cast<double>(t.ax));
  t.ly = static_cast<float>(ti.ay - static_cast<double>(t.ay));
  t.lz = static_cast<float>(ti.az - static_cast<double>(t.az));
  const double ai[3] = {ti.ax, ti.ay, ti.az};
  const float eps = static_cast<float>(kEpsPair * scale * scale);

  // stretching: G mode, and the row's box for the far test
  bool g64 = false;
  double cen[3] = {0, 0, 0}, half[3] = {0, 0, 0}, smax = 0.0;
  if constexpr (S::str) {
    if constexpr (!S::pse && (S::vort || S::ens)) {
      g64 = true;
    } else {
      g64 = a.g64_mode == VPM_G64_ALWAYS;
      if (a.g64_mode == VPM_G64_AUTO) g64 = coherent_wave<1>(&ti, &valid);
    }
    g64 = __builtin_amdgcn_readfirstlane(static_cast<int>(g64)) != 0;
    const double p[3] = {X, Y, Z};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const double lo = wave_min(valid ? p[q] : INFINITY), hi = wave_max(valid ? p[q] : -INFINITY);
      cen[q] = 0.5 * (lo + hi);
      half[q] = 0.5 * (hi - lo);
    }
    smax = wave_max(valid ? ti.s * scale : 0.0);
  }

  float part[kNAcc];
  double tot[kNAcc], gsum[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < kNAcc; ++q) {
    part[q] = 0.0f;
    tot[q] = 0.0;
  }
  PairConst<float> kc{1.5f, 7.5f, 2.2f, 3.0f, 2.5f};  // in VGPRs (see PairConst)
  asm volatile("" : "+v"(kc.c15), "+v"(kc.c75), "+v"(kc.c22), "+v"(kc.c3));

  const int nchunk = (a.n + kChunk32 - 1) / kChunk32;
  const int parts = splits * kRowWaves;
  for (int c = static_cast<int>(blockIdx.y) * kRowWaves + wave; c < nchunk; c += parts) {
    const scalar_double_t* box =
        (const scalar_double_t*)(box_ + static_cast<int64_t>(c) * kBox32);
    t.x = static_cast<float>(X - box[0]);
    t.y = static_cast<float>(Y - box[1]);
    t.z = static_cast<float>(Z - box[2]);
    const int j0 = c * kChunk32;
    const far_float_t* rec =
        (const far_float_t*)(rec_ + static_cast<int64_t>(j0) * R::kStride);
    bool fp64 = g64;
    if constexpr (S::str) {
      if (g64 && c != row) {
        double gap2 = 0.0;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const double gp = fmax(fabs(box[q] - cen[q]) - half[q] - box[3 + q], 0.0);
          gap2 += gp * gp;
        }
        const double lim = kFarGap32 * fmax(smax, box[6]);
        fp64 = __builtin_amdgcn_readfirstlane(static_cast<int>(!(gap2 > lim * lim))) != 0;
      }
    }
    auto load = [&](float* b, int q, int cnt) {
#pragma unroll
      for (int u = 0; u < kGroup32 * R::kStride; ++u)
        if (u < cnt * R::kStride) b[u] = rec[q * R::kStride + u];
    };
    if (S::str && (c == row || fp64)) {
      if constexpr (S::str) {
        // the row's own chunk, and near chunks of FP64 rows: valid sources only
        const int cnt = a.n - j0 < kChunk32 ? a.n - j0 : kChunk32;
        const scalar_double_t* str =
            (const scalar_double_t*)(reinterpret_cast<const double*>(a.src + j0));
        if (fp64) {
          const bool own = c == row;
#pragma unroll 2
          for (int q = 0; q < cnt; ++q) {
            float f[R::kStride];
#pragma unroll
            for (int u = 0; u < R::kStride; ++u) f[u] = rec[q * R::kStride + u];
            const double aj[3] = {str[q * 8 + 3], str[q * 8 + 4], str[q * 8 + 5]};
            pair32<OUT, UNIF, true>(part, gsum, t, f, aj, ai, eps, kc, own && q == lane);
          }
        } else {
#pragma unroll 1
          for (int q = 0; q < cnt; ++q) {
            float f[R::kStride];
#pragma unroll
            for (int u = 0; u < R::kStride; ++u) f[u] = rec[q * R::kStride + u];
            pair32<OUT, UNIF, false>(part, gsum, t, f, nullptr, ai, eps, kc, q == lane);
          }
        }
      }
    } else {
      // groups of four in two register buffers: a group's loads issue after
      // the first pair of the one before it (scalar loads return out of
      // order, so a wait covers every load in flight); the last reads one
      // group of padding
      float bA[kGroup32 * R::kStride], bB[kGroup32 * R::kStride];
      auto group = [&](const float* b, float* nb, int qn) {
        pair32<OUT, UNIF, false>(part, gsum, t, b, nullptr, ai, eps, kc, false);
        __builtin_amdgcn_sched_barrier(0);
        load(nb, qn, kGroup32);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 1; u < kGroup32; ++u)
          pair32<OUT, UNIF, false>(part, gsum, t, b + u * R::kStride, nullptr, ai, eps, kc, false);
      };
      load(bA, 0, kGroup32);
#pragma unroll 1
      for (int q = 0; q < kChunk32; q += 2 * kGroup32) {
        group(bA, bB, q + kGroup32);
        group(bB, bA, q + 2 * kGroup32);
      }
    }
#pragma unroll
    for (int q = 0; q < kNAcc; ++q)
      if (S::used(q)) {
        tot[q] += static_cast<double>(part[q]);
        part[q] = 0.0f;
      }
    if constexpr (S::str) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        gsum[q] += static_cast<double>(part[kG + q]);
        part[kG + q] = 0.0f;
      }
    }
  }

  // the waves' totals, in wave order
#pragma unroll
  for (int q = 0; q < kNAcc; ++q)
    if (S::used(q)) red[wave][S::packed(q)][lane] = tot[q];
  if constexpr (S::str) {
#pragma unroll
    for (int q = 0; q < 3; ++q) red[wave][S::nacc + q][lane] = gsum[q];
  }
  __syncthreads();
  for (int q = wave; q < NS; q += kRowWaves) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) s += red[w][q][lane];
    if (a.part)
      a.part[(static_cast<int64_t>(blockIdx.y) * NS + q) * a.pld + kt] = s;
    else
      red[0][q][lane] = s;  // read by this wave only, above
  }
  if (a.part) return;
  __syncthreads();
  if (wave != 0) return;
  double T[kNAcc], G[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < kNAcc; ++q) T[q] = S::used(q) ? red[0][S::packed(q)][lane] : 0.0;
  if constexpr (S::str) {
#pragma unroll
    for (int q = 0; q < 3; ++q) G[q] = red[0][S::nacc + q][lane];
  }
  double ens = 0.0;
  if (valid) ens = store_target<OUT, true>(a, ti, a.perm ? a.perm[kt] : kt, T, G, scale);
  if constexpr (S::ens) {
    ens = wave_sum(ens);
    if (lane == 0) a.ens_part[row] = ens;
  }
}

int nslots(unsigned mask) {
  int c = 0;
  for (unsigned b = 1; b <= VPM_OUT_ENSTROPHY; b <<= 1) c += (mask & b) ? 3 : 0;
  return c + ((mask & VPM_OUT_STRETCH) ? 3 : 0);
}

template <unsigned OUT, bool UNIF>
int launch(FusedArgs a, float* rec, double* box, hipStream_t st, int* nblocks) {
  using R = Rec32<OUT, UNIF>;
  const int rows = static_cast<int>(ceil_div(a.n, kRow));
  const int chunks = static_cast<int>(ceil_div(a.n, kChunk32));
  const size_t per = static_cast<size_t>(Slots<OUT>::nslot) * rows * kRow * sizeof(double);
  int k = std::min(row_splits(rows, a.n), std::max(1, chunks / kRowWaves));
  if (a.max_splits > 0) k = std::min(k, a.max_splits);
  if (!a.part || a.part_cap / per < 2) k = 1;
  else k = static_cast<int>(std::min<size_t>(k, a.part_cap / per));
  if (k == 1) a.part = nullptr;
  a.pld = static_cast<int64_t>(rows) * kRow;
  hipLaunchKernelGGL(row32_records_kernel, dim3(chunks), dim3(kChunk32), 0, st, a.src, a.n,
                     R::kStride, R::kLoAt, UNIF ? 1 : 0, rec, box);
  VPM_LAUNCH_CHECK("row32_records_kernel");
  hipLaunchKernelGGL((row32_kernel<OUT, UNIF>), dim3(rows, k), dim3(kRowBlock), 0, st, a, k, rec,
                     box);
  VPM_LAUNCH_CHECK("row32_kernel");
  *nblocks = rows;
  if (k > 1) {
    const int rb = static_cast<int>(ceil_div(a.n, 256));
    hipLaunchKernelGGL((split_reduce_kernel<OUT, true>), dim3(rb), dim3(256), 0, st, a, k);
    VPM_LAUNCH_CHECK("split_reduce_kernel");
    *nblocks = rb;
  }
  return VPM_OK;
}

}  // namespace

// Records of whole chunks, and one group read ahead past the last.
size_t row32_record_bytes(int64_t n) {
  return (static_cast<size_t>(ceil_div(n > 0 ? n : 1, kChunk32)) * kChunk32 + kGroup32) *
         kStride32 * sizeof(float);
}

size_t row32_box_bytes(int64_t n) {
  return static_cast<size_t>(ceil_div(n > 0 ? n : 1, kChunk32)) * kBox32 * sizeof(double);
}

size_t row32_split_bytes(int64_t n, unsigned mask) {
  const int64_t rows = row_count(n);
  const int k = row_splits(rows, n);
  return k > 1 ? static_cast<size_t>(k) * nslots(mask) * rows * kRow * sizeof(double) : 0;
}

int row32_run(const FusedArgs& a, unsigned mask, bool unif, float* rec, double* box,
              hipStream_t st, int* nblocks) {
  switch (mask | (unif ? 32u : 0u)) {
#define VPM_ROW32(M, U)      \
  case (M) | ((U) ? 32u : 0u): \
    return launch<M, U>(a, rec, box, st, nblocks);
    VPM_ROW32(1u, true) VPM_ROW32(2u, true) VPM_ROW32(4u, true) VPM_ROW32(8u, true)
    VPM_ROW32(16u, true) VPM_ROW32(24u, true)
    VPM_ROW32(1u, false) VPM_ROW32(2u, false) VPM_ROW32(3u, false) VPM_ROW32(4u, false)
    VPM_ROW32(7u, false) VPM_ROW32(8u, false) VPM_ROW32(16u, false) VPM_ROW32(24u, false)
    VPM_ROW32(27u, false) VPM_ROW32(31u, false)
#undef VPM_ROW32
    default:
      return fail(VPM_ERR_ARG, "row32: output set has the far-field moment form");
  }
}

}  // namespace vpm
