// FP32-compensated pair sums over rows of 64 sorted targets.
//
// A workgroup owns one row; its eight waves take the source chunks in turn
// (chunk c goes to part c mod parts, over the waves and the source splits), so
// a row's few near chunks spread over the waves.  Every lane of a wave pairs
// with the same source, so the sources come through scalar loads from FP32
// records relative to their chunk's centre, and enter the pair instructions
// as scalar operands: no LDS staging, no barrier in the sweep.  (The tiled
// kernels read up to 48 bytes per source and wave from LDS, 3 x 8 clocks of
// the CU's LDS return path against about 18 clocks of FP32 issue: LDS bound
// them.)  The target's offset to the chunk centre comes from FP64 positions
// once per chunk; FP32 partials of a chunk are folded into FP64 totals, which
// wait in LDS meanwhile.
//
// Far chunks (gap between the row's and the chunk's boxes above kFarGap32
// times the larger radius) of sets with stretching, another output and a
// uniform radius take the moment form (pair_far).  Stretching: rows of coherent
// strengths (coherent_wave) take the sum of g alpha_j and the triple product
// in FP64, the others in FP32, as in the tiled kernels (vpm_fused.hip, which
// also measures why); sets with vorticity or enstrophy and without PSE sum in
// FP64 in every row.  The moment form is FP32 in every row.
//
// With s = sigma_ij, D = r^2 + s^2, t = D^-1/2 and w = s^2 t^2 no reciprocal
// of s is needed: (rho^2 + 2.5) / (A^5/2 s^3) = t^3 (1 + 1.5 w) and so on
// (vpm_plain.hip).
//
// Bound: FP32 issue (velocity alone 2.45e12 pairs/s, 1.55 wave64 instructions
// per clock and CU; the moment form 1.8e12).  Tiled kernels -> here, per call.
// N = 100,000: velocity 4.80 -> 4.17 ms, with per-particle radii 6.80 -> 4.78;
// stretching of a ring 8.92 -> 7.99, 10.9 -> 8.60; PSE 5.81 -> 4.92, 6.75 ->
// 5.4; vorticity + enstrophy 4.97 -> 4.73, 7.15 -> 6.15; all five with
// per-particle radii 15.7 -> 14.3 (cloud), 18.8 -> 17.6 (ring).  Velocity +
// stretching: cloud of 2^20 614 -> 605, of 20,000 0.448 -> 0.328, ring of
// 131,072 12.8 -> 11.1; with PSE: ring of 131,072 15.7 -> 13.1, leapfrogging
// rings of 65,536 4.30 -> 3.49.

#include "vpm_row32.h"

#include <algorithm>

#include "vpm_rows.h"

namespace vpm {

namespace {

constexpr int kMinChunk32 = 64, kMaxChunk32 = 128;  // sources per chunk (Rec32)
constexpr int kStride32 = 12;     // most floats per record
constexpr int kMaxGroup32 = 4;    // records per group of scalar loads (Rec32)
constexpr int kBox32 = 8;         // doubles per chunk box: centre, half-extent, largest radius
constexpr double kFarGap32 = 4.0;
// Waves per SIMD the registers must allow: 73 VGPRs for velocity + stretching
// (cloud of 2^20: 605 ms; 641 at five waves, 687 at eight, where the records
// spill scalar registers); eight for the stretching alone, whose records and
// sums are the smallest (cloud of 65,536 with a uniform radius 2.95 -> 2.81 ms,
// ring 3.94 -> 3.81).
template <unsigned OUT>
constexpr int kRow32Waves = OUT == VPM_OUT_STRETCH ? 8 : 6;

// Record layout: offset (3), strength (3); then with the moment form the
// moment alpha x offset (3; three times it with PSE, pair_far), with
// per-particle radii sigma/2 and sigma^-2, with vorticity sigma^-3 behind them
// (with PSE last); with PSE the low parts alpha - fp32(alpha).  Lengths in
// units of a uniform radius; with per-particle radii as they are: any one
// particle's radius may be far from the others', and the powers of t leave
// FP32 where distances are 1e8 units.
// Two groups are in registers at once: of four records, or of two where a
// record has twelve floats and four would spill scalar registers (velocity +
// stretching + PSE, cloud of 131,072: 11.4 against 12.5 ms, ring 13.4 against
// 13.8).  Chunks of 128 sources halve the moment form's set-up and fold per chunk;
// with the LES outputs 64 keep the vorticity's partials as short as they were
// (rel-L2 1.0e-7 against 1.5e-7 on a ring of 20,000), and in a batch every
// output's, whose tiled launch folds 64 (velocity of 24 sets, mean rel-L2
// 1.14e-7 with 64, 1.56e-7 with 128, tiled 1.45e-7; a stage with PSE 4.29 and
// 4.34 ms, tiled 7.37).
template <unsigned OUT, bool UNIF, bool BATCH = false>
struct Rec32 {
  static constexpr bool kLo = OUT & VPM_OUT_PSE;
  // Far chunks take the moment form, in FP32 in every row.  Without it rows
  // that sum the stretching in FP64 per pair do so on every chunk: FP32 sums of
  // g alpha_j leave 1e-7 of |alpha_i| |G|, and along a tube of parallel
  // strengths nothing else is left.  FP64 everywhere costs a ring of 100,000
  // with per-particle radii 8.6 ms instead of 7.3 (stretching; tiled kernels
  // 10.9), a cloud, whose rows are not coherent, nothing.
  static constexpr bool kMoment = UNIF && (OUT & VPM_OUT_STRETCH) && OUT != VPM_OUT_STRETCH;
  static constexpr bool kE3 = kMoment && kLo;
  static constexpr int kLoAt = kMoment ? 9 : UNIF ? 6 : 8;
  static constexpr int kIs3At = kLo ? 11 : 8;
  static constexpr bool kOwnVort = !UNIF && (OUT & VPM_OUT_VORT);
  static constexpr int kStride = kLo ? 12 : kMoment || kOwnVort ? 9 : UNIF ? 6 : 8;
  static constexpr int kGroup = kLo ? 2 : kMaxGroup32;
  static constexpr int kNear = kLo ? 4 : 2;  // sources in flight in the FP64 loop
  static constexpr int kChunk =
      kMoment && !BATCH && !(OUT & (VPM_OUT_VORT | VPM_OUT_ENSTROPHY)) ? kMaxChunk32 : kMinChunk32;
};

__device__ __forceinline__ double held(double v) {  // rounded here, not fused into its use
  asm volatile("" : "+v"(v));
  return v;
}

// The records and box of chunk c of a set of n sorted particles, by one
// workgroup of kChunk lanes; rec and box_ are the set's.  Lanes past n write
// zero-strength padding far away, which adds exactly 0.  The box is that of
// the finite coordinates: a particle at infinity keeps an infinite offset (PSE
// and vorticity weigh it 0) and leaves its chunk's others theirs.
template <unsigned OUT, bool UNIF, bool BATCH>
__device__ __forceinline__ void row32_records(const Src8* __restrict__ src, int n, int c,
                                              float* __restrict__ rec, double* __restrict__ box_) {
  using R = Rec32<OUT, UNIF, BATCH>;
  __shared__ double red[7][R::kChunk / 64];
  const int k = c * R::kChunk + static_cast<int>(threadIdx.x);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool ok = k < n;
  const double scale = UNIF ? 1.0 / src[0].s : 1.0;
  Src8 g{};
  if (ok) g = src[k];
  const double p[3] = {held(g.x * scale), held(g.y * scale), held(g.z * scale)};
  const double sig = g.s * scale;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const bool in = ok && isfinite(p[q]);
    const double lo = wave_min(in ? p[q] : INFINITY), hi = wave_max(in ? p[q] : -INFINITY);
    if (lane == 0) {
      red[q][wave] = lo;
      red[3 + q][wave] = hi;
    }
  }
  const double big = wave_max(ok ? sig : 0.0);
  if (lane == 0) red[6][wave] = big;
  __syncthreads();
  double cen[3];
  double* box = box_ + static_cast<int64_t>(c) * kBox32;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    double lo = red[q][0], hi = red[3 + q][0];
#pragma unroll
    for (int w = 1; w < R::kChunk / 64; ++w) {
      lo = fmin(lo, red[q][w]);
      hi = fmax(hi, red[3 + q][w]);
    }
    cen[q] = lo <= hi ? 0.5 * (lo + hi) : 0.0;
    if (threadIdx.x == 0) {
      box[q] = cen[q];
      box[3 + q] = lo <= hi ? 0.5 * (hi - lo) : 0.0;
    }
  }
  if (threadIdx.x == 0) {
    double m = red[6][0];
#pragma unroll
    for (int w = 1; w < R::kChunk / 64; ++w) m = fmax(m, red[6][w]);
    box[6] = m;
    box[7] = 0.0;
  }
  float* r = rec + static_cast<int64_t>(k) * R::kStride;
  const double x = p[0] - cen[0], y = p[1] - cen[1], z = p[2] - cen[2];
  const float ax = static_cast<float>(g.ax), ay = static_cast<float>(g.ay),
              az = static_cast<float>(g.az);
  r[0] = ok ? static_cast<float>(x) : 1e18f;
  r[1] = ok ? static_cast<float>(y) : 1e18f;
  r[2] = ok ? static_cast<float>(z) : 1e18f;
  r[3] = ax;
  r[4] = ay;
  r[5] = az;
  if constexpr (R::kMoment) {
    constexpr double ms = R::kE3 ? 3.0 : 1.0;
    r[6] = ok ? static_cast<float>(ms * (g.ay * z - g.az * y)) : 0.0f;
    r[7] = ok ? static_cast<float>(ms * (g.az * x - g.ax * z)) : 0.0f;
    r[8] = ok ? static_cast<float>(ms * (g.ax * y - g.ay * x)) : 0.0f;
  } else if constexpr (!UNIF) {
    r[6] = ok ? static_cast<float>(0.5 * sig) : 0.5f;
    r[7] = ok ? static_cast<float>(1.0 / (sig * sig)) : 1.0f;
    if constexpr (R::kOwnVort && !R::kLo)
      r[R::kIs3At] = ok ? static_cast<float>(1.0 / (sig * sig * sig)) : 1.0f;
  }
  if constexpr (R::kLo) {
    r[R::kLoAt] = static_cast<float>(g.ax - static_cast<double>(ax));
    r[R::kLoAt + 1] = static_cast<float>(g.ay - static_cast<double>(ay));
    r[R::kLoAt + 2] = static_cast<float>(g.az - static_cast<double>(az));
    for (int q = R::kLoAt + 3; q < R::kStride; ++q) r[q] = 0.0f;
    if constexpr (R::kOwnVort)
      r[R::kIs3At] = ok ? static_cast<float>(1.0 / (sig * sig * sig)) : 1.0f;
  }
}

template <unsigned OUT, bool UNIF>
__global__ __launch_bounds__((Rec32<OUT, UNIF>::kChunk)) void row32_records_kernel(
    const Src8* __restrict__ src, int n, float* __restrict__ rec, double* __restrict__ box) {
  row32_records<OUT, UNIF, false>(src, n, static_cast<int>(blockIdx.x), rec, box);
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
    float cx, cy, cz, e = 0.0f;
    if constexpr (G64 && S::str) {
      const double rx = dx, ry = dy, rz = dz;
      const double qx = ry * aj[2] - rz * aj[1];
      const double qy = rz * aj[0] - rx * aj[2];
      const double qz = rx * aj[1] - ry * aj[0];
      e = static_cast<float>(ai[0] * qx + ai[1] * qy + ai[2] * qz);
      cx = static_cast<float>(qx);
      cy = static_cast<float>(qy);
      cz = static_cast<float>(qz);
    } else {
      cx = dy * f[5] - dz * f[4];
      cy = dz * f[3] - dx * f[5];
      cz = dx * f[4] - dy * f[3];
    }
    if constexpr (S::vel) {
      acc[kU + 0] += g * cx;
      acc[kU + 1] += g * cy;
      acc[kU + 2] += g * cz;
    }
    if constexpr (S::str) {
      const float gG = self ? 0.0f : g;
      if constexpr (G64) {
        const double gd = gG;
        g64[0] = fma(gd, aj[0], g64[0]);
        g64[1] = fma(gd, aj[1], g64[1]);
        g64[2] = fma(gd, aj[2], g64[2]);
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
    float v;
    if constexpr (UNIF) {
      v = (t3 * t3) * t3;
    } else {
      // t2 carries the root's and its own rounding, the ninth power of t 4.5 of
      // them (PSE of rings and clouds with per-particle radii, rel-L2 1.13
      // times the tiled kernels' without this, 0.8 with)
      // 1 - D t2, exact but for one rounding (of no weight at infinity)
      const float r = fminf(__builtin_fmaf(-D, t2, 1.0f), 1.0f);
      v = ((s * t3) * (w * w * w)) * __builtin_fmaf(k.c45, r, 1.0f);
    }
    acc[kP + 0] += v * ((f[3] - t.ax) + (lo[0] - t.lx));
    acc[kP + 1] += v * ((f[4] - t.ay) + (lo[1] - t.ly));
    acc[kP + 2] += v * ((f[5] - t.az) + (lo[2] - t.lz));
  }
  if constexpr (S::vort) {
    float v;
    if constexpr (UNIF) {
      v = t3 * (t2 * t2);
    } else {  // sigma_j, not sigma_ij (ParticlesPhysicsCuda.py:323,334-337)
      // in units of sigma_j: near sources 1 + r^2 / sigma_j^2 carries less of
      // the factors' rounding than r^2 + sigma_j^2 (rel-L2 1.04 times as large)
      const float q1 = __builtin_amdgcn_rsqf(__builtin_fmaf(r2, f[7], 1.0f));
      const float q2 = q1 * q1;
      v = ((q2 * q2) * (q2 * q1)) * f[Rec32<OUT, UNIF>::kIs3At];
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

// The far-field moment form of the stretching with a uniform radius, with or
// without the velocity (pair_moment in vpm_fused.hip derives and measures it):
// 29 instructions per pair with it, p = alpha_i x x_i (three times it with
// PSE).
template <unsigned OUT>
__device__ __forceinline__ void pair_far(float* acc, const Tgt32& t, const float* p, const float* f,
                                         const PairConst<float>& k) {
  using S = Slots<OUT>;
  const float dx = t.x - f[0], dy = t.y - f[1], dz = t.z - f[2];
  const float D = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, 1.0f)));
  const float t1 = __builtin_amdgcn_rsqf(D);
  const float t2 = t1 * t1;
  const float t3 = t2 * t1;
  const float t5 = t3 * t2;
  const float g = __builtin_fmaf(k.c15, t5, t3);
  acc[kG + 0] = __builtin_fmaf(g, f[3], acc[kG + 0]);
  acc[kG + 1] = __builtin_fmaf(g, f[4], acc[kG + 1]);
  acc[kG + 2] = __builtin_fmaf(g, f[5], acc[kG + 2]);
  if constexpr (S::vel) {
    acc[kH + 0] = __builtin_fmaf(g, f[6], acc[kH + 0]);
    acc[kH + 1] = __builtin_fmaf(g, f[7], acc[kH + 1]);
    acc[kH + 2] = __builtin_fmaf(g, f[8], acc[kH + 2]);
  }
  float e = f[3] * p[0];
  e = __builtin_fmaf(f[4], p[1], e);
  e = __builtin_fmaf(f[5], p[2], e);
  e = __builtin_fmaf(t.ax, f[6], e);
  e = __builtin_fmaf(t.ay, f[7], e);
  e = __builtin_fmaf(t.az, f[8], e);
  const float t7 = t5 * t2;
  float w;
  if constexpr (Rec32<OUT, true>::kE3)
    w = __builtin_fmaf(k.c25, t7, t5) * e;
  else
    w = t5 * __builtin_fmaf(k.c75, t2, k.c3) * e;
  acc[kSd + 0] = __builtin_fmaf(w, dx, acc[kSd + 0]);
  acc[kSd + 1] = __builtin_fmaf(w, dy, acc[kSd + 1]);
  acc[kSd + 2] = __builtin_fmaf(w, dz, acc[kSd + 2]);
  if constexpr (S::vort) {
    acc[kW + 0] = __builtin_fmaf(t7, f[3], acc[kW + 0]);
    acc[kW + 1] = __builtin_fmaf(t7, f[4], acc[kW + 1]);
    acc[kW + 2] = __builtin_fmaf(t7, f[5], acc[kW + 2]);
  }
  if constexpr (S::ens) {
    const float en = __builtin_fmaf(k.c22, t3, t1);
    acc[kE + 0] = __builtin_fmaf(en, f[3], acc[kE + 0]);
    acc[kE + 1] = __builtin_fmaf(en, f[4], acc[kE + 1]);
    acc[kE + 2] = __builtin_fmaf(en, f[5], acc[kE + 2]);
  }
  if constexpr (S::pse) {  // sum t9 alpha_j - alpha_i sum t9, the second part per chunk
    const float t9 = t7 * t2;
    acc[kP + 0] = __builtin_fmaf(t9, f[3], acc[kP + 0]);
    acc[kP + 1] = __builtin_fmaf(t9, f[4], acc[kP + 1]);
    acc[kP + 2] = __builtin_fmaf(t9, f[5], acc[kP + 2]);
    acc[kT9] += t9;
  }
}

// Rows of many sets in one launch (24 rings and clouds of 2,048 to 32,768
// particles, RK4 step with PSE and LES: 29.2 ms with persistent 256-target
// items, whose one round the largest sets' items outlasted, 17.3 ms here):
// workgroup w takes row w % rows_per_item of
// item w / rows_per_item (an item is a target block of a set; the list runs
// from the largest set to the smallest, and the dispatcher hands out
// workgroups in that order).  Rows past the set's end leave at once, with a
// zero enstrophy partial.
struct Row32Item {
  int set, off, n, row;
};

__device__ __forceinline__ bool row32_item(const Row32Batch& b, int w, Row32Item* it) {
  const int item = w / b.rows_per_item;
  it->set = b.item_set[item];
  it->off = b.set_off[it->set];
  it->n = b.set_off[it->set + 1] - it->off;
  it->row = b.item_block[item] * b.rows_per_item + w % b.rows_per_item;
  return it->row * kRow < it->n;
}

// grid (rows, splits); batched: (items * rows_per_item, splits).  (One kernel
// with the set picked at its top: as a device function called from two kernels
// the same body took up to 46 more VGPRs, into scratch.)
template <unsigned OUT, bool UNIF, bool BATCH>
__global__ __launch_bounds__(kRowBlock, kRow32Waves<OUT>) void row32_kernel(
    FusedArgs a, Row32Batch b, int splits, const float* __restrict__ rec_,
    const double* __restrict__ box_) {
  const int split = static_cast<int>(blockIdx.y);
  int n = a.n, row = static_cast<int>(blockIdx.x);
  const Src8* src = a.src;
  const int* perm = a.perm;
  double* part_out =
      a.part ? a.part + static_cast<int64_t>(split) * Slots<OUT>::nslot * a.pld : nullptr;
  if constexpr (BATCH) {
    Row32Item it;
    if (!row32_item(b, row, &it)) {
      if (threadIdx.x == 0 && split == 0) a.ens_part[row] = 0.0;
      return;
    }
    const int64_t c0 = b.chunk0[it.set];
    rec_ = b.rec + c0 * Rec32<OUT, UNIF, BATCH>::kChunk * Rec32<OUT, UNIF, BATCH>::kStride;
    box_ = b.box + c0 * kBox32;
    n = it.n;
    row = it.row;
    src += it.off;
    perm += it.off;
    if (part_out) part_out += it.off;
  }
  using S = Slots<OUT>;
  using R = Rec32<OUT, UNIF, BATCH>;
  constexpr int NS = S::nslot, CH = R::kChunk;
  // FP64 totals of each wave's share (kept here, not in registers: they are
  // touched once per chunk) and, at the end, their sums
  __shared__ double tot[kRowWaves][NS][kRow];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kt = row * kRow + lane;
  const bool valid = kt < n;
  const double scale = UNIF ? 1.0 / src[0].s : 1.0;
  Src8 ti{0, 0, 0, 0, 0, 0, 1, 0};
  if (valid) ti = src[kt];
  const double X = held(ti.x * scale), Y = held(ti.y * scale), Z = held(ti.z * scale);
  Tgt32 t;
  t.ax = static_cast<float>(ti.ax);
  t.ay = static_cast<float>(ti.ay);
  t.az = static_cast<float>(ti.az);
  t.hs = static_cast<float>(0.5 * ti.s * scale);
  t.lx = static_cast<float>(ti.ax - static_cast<double>(t.ax));
  t.ly = static_cast<float>(ti.ay - static_cast<double>(t.ay));
  t.lz = static_cast<float>(ti.az - static_cast<double>(t.az));
  const float eps = static_cast<float>(kEpsPair * scale * scale);
  // The target's FP64 record is read again where it is needed (FP64 chunks,
  // the epilogue) instead of staying in registers through the sweep.
  auto target = [&]() {
    int k = valid ? kt : row * kRow;
    asm volatile("" : "+v"(k));
    return src[k];
  };

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
  }
  if constexpr (R::kMoment) {
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
#pragma unroll
  for (int q = 0; q < kNAcc; ++q) part[q] = 0.0f;
#pragma unroll
  for (int q = 0; q < NS; ++q) tot[wave][q][lane] = 0.0;
  PairConst<float> kc{1.5f, 7.5f, 2.2f, 3.0f, 2.5f, 4.5f};  // in VGPRs (see PairConst)
  asm volatile("" : "+v"(kc.c15), "+v"(kc.c75), "+v"(kc.c22), "+v"(kc.c3), "+v"(kc.c25));
  if constexpr (!UNIF) asm volatile("" : "+v"(kc.c45));

  const int nchunk = (n + CH - 1) / CH;
  const int parts = splits * kRowWaves;
  const int own = row * kRow / CH;          // the chunk that holds the row
  uint64_t near = 0;                        // this wave's next 64 chunks near the row
  int seen = 0;
  for (int c = split * kRowWaves + wave; c < nchunk; c += parts, ++seen) {
    bool is_near = true;
    if constexpr (R::kMoment) {
      // far tests for 64 of the wave's chunks at a time, one per lane
      if ((seen & 63) == 0) {
        const int64_t cc = c + static_cast<int64_t>(lane) * parts;
        bool nr = false;
        if (cc < nchunk) {
          const double* box = box_ + cc * kBox32;
          double gap2 = 0.0;
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            const double gp = fmax(fabs(box[q] - cen[q]) - half[q] - box[3 + q], 0.0);
            gap2 += gp * gp;
          }
          const double lim = kFarGap32 * fmax(smax, box[6]);
          nr = !(gap2 > lim * lim);
        }
        near = __ballot(nr);
      }
      is_near = ((near >> (seen & 63)) & 1u) != 0;
    }
    const bool fp64 = g64 && is_near;
    const scalar_double_t* box =
        (const scalar_double_t*)(box_ + static_cast<int64_t>(c) * kBox32);
    t.x = static_cast<float>(X - box[0]);
    t.y = static_cast<float>(Y - box[1]);
    t.z = static_cast<float>(Z - box[2]);
    const int j0 = c * CH;
    const far_float_t* rec =
        (const far_float_t*)(rec_ + static_cast<int64_t>(j0) * R::kStride);
    auto load1 = [&](float* f, int q) {
#pragma unroll
      for (int u = 0; u < R::kStride; ++u) f[u] = rec[q * R::kStride + u];
    };
    // Groups of records in two register buffers: a group's loads issue
    // after the first pair of the one before it (scalar loads return out of
    // order, so a wait covers every load in flight); the last reads one group
    // of padding.
    auto stream = [&](auto pair) {
      float bA[R::kGroup * R::kStride], bB[R::kGroup * R::kStride];
      auto load = [&](float* b, int q) {
#pragma unroll
        for (int u = 0; u < R::kGroup * R::kStride; ++u) b[u] = rec[q * R::kStride + u];
      };
      auto group = [&](const float* b, float* nb, int qn) {
        pair(b, qn - R::kGroup);
        __builtin_amdgcn_sched_barrier(0);
        load(nb, qn);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 1; u < R::kGroup; ++u) pair(b + u * R::kStride, qn - R::kGroup + u);
      };
      load(bA, 0);
#pragma unroll 1
      for (int q = 0; q < CH; q += 2 * R::kGroup) {
        group(bA, bB, q + R::kGroup);
        group(bB, bA, q + 2 * R::kGroup);
      }
    };
    double g64s[3] = {0.0, 0.0, 0.0};
    if (S::str && (fp64 || c == own)) {
      if constexpr (S::str) {
        const int cnt = n - j0 < CH ? n - j0 : CH;
        const int self = c == own ? lane + (row * kRow - j0) : -1;
        const scalar_double_t* str =
            (const scalar_double_t*)(reinterpret_cast<const double*>(src + j0));
        if (fp64) {  // valid sources only
          const Src8 tr = target();
          const double ai[3] = {tr.ax, tr.ay, tr.az};
#pragma unroll R::kNear
          for (int q = 0; q < cnt; ++q) {
            float f[R::kStride];
            load1(f, q);
            const double aj[3] = {str[q * 8 + 3], str[q * 8 + 4], str[q * 8 + 5]};
            pair32<OUT, UNIF, true>(part, g64s, t, f, aj, ai, eps, kc, q == self);
          }
        } else {
          // the row's own chunk, streamed like the others: one record at a time
          // each pair waited for its load, and the wave with this chunk held up
          // its row (velocity + stretching, cloud of 9,000: 113 -> 110 us)
          stream([&](const float* f, int q) {
            pair32<OUT, UNIF, false>(part, g64s, t, f, nullptr, nullptr, eps, kc, q == self);
          });
        }
      }
    } else if (!R::kMoment || is_near) {
      stream([&](const float* f, int) {
        pair32<OUT, UNIF, false>(part, g64s, t, f, nullptr, nullptr, eps, kc, false);
      });
    } else if constexpr (R::kMoment) {
      constexpr float es = R::kE3 ? 3.0f : 1.0f;
      const float p[3] = {es * (t.ay * t.z - t.az * t.y), es * (t.az * t.x - t.ax * t.z),
                          es * (t.ax * t.y - t.ay * t.x)};
      stream([&](const float* f, int) { pair_far<OUT>(part, t, p, f, kc); });
      if constexpr (S::vel) {  // u += x_i x G + H of the chunk, in FP64
        const double x = X - box[0], y = Y - box[1], z = Z - box[2];
        const double gx = part[kG + 0], gy = part[kG + 1], gz = part[kG + 2];
        constexpr double hs = R::kE3 ? 1.0 / 3.0 : 1.0;
        double* u = &tot[wave][0][lane];
        u[0] += (y * gz - z * gy) + static_cast<double>(part[kH + 0]) * hs;
        u[kRow] += (z * gx - x * gz) + static_cast<double>(part[kH + 1]) * hs;
        u[2 * kRow] += (x * gy - y * gx) + static_cast<double>(part[kH + 2]) * hs;
        part[kH + 0] = part[kH + 1] = part[kH + 2] = 0.0f;
      }
      if constexpr (S::pse) {
        part[kP + 0] = __builtin_fmaf(-t.ax, part[kT9], part[kP + 0]);
        part[kP + 1] = __builtin_fmaf(-t.ay, part[kT9], part[kP + 1]);
        part[kP + 2] = __builtin_fmaf(-t.az, part[kT9], part[kP + 2]);
        part[kT9] = 0.0f;
      }
    }
#pragma unroll
    for (int q = 0; q < kNAcc; ++q)
      if (S::used(q)) {
        tot[wave][S::packed(q)][lane] += static_cast<double>(part[q]);
        part[q] = 0.0f;
      }
    if constexpr (S::str) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        tot[wave][S::nacc + q][lane] += g64s[q] + static_cast<double>(part[kG + q]);
        part[kG + q] = 0.0f;
      }
    }
  }

  // the waves' totals, in wave order
  __syncthreads();
  for (int q = wave; q < NS; q += kRowWaves) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) s += tot[w][q][lane];
    if (!part_out)
      tot[0][q][lane] = s;  // slot q is read by this wave only, above
    else if (valid)
      part_out[q * a.pld + kt] = s;
  }
  if (part_out) return;
  __syncthreads();
  if (wave != 0) return;
  double T[kNAcc], G[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < kNAcc; ++q) T[q] = S::used(q) ? tot[0][S::packed(q)][lane] : 0.0;
  if constexpr (S::str) {
#pragma unroll
    for (int q = 0; q < 3; ++q) G[q] = tot[0][S::nacc + q][lane];
  }
  double ens = 0.0;
  if (valid) ens = store_target<OUT, UNIF>(a, target(), perm ? perm[kt] : kt, T, G, scale);
  if constexpr (S::ens) {
    ens = wave_sum(ens);
    if (lane == 0) a.ens_part[blockIdx.x] = ens;
  }
}

// set_chunk0[s] = chunks of the sets before s; set_chunk0[S] = all.
__global__ __launch_bounds__(1024) void row32_chunks_kernel(const int* __restrict__ off, int nsets,
                                                            int ch, int* __restrict__ chunk0) {
  __shared__ int part[1024];
  const int t = threadIdx.x;
  const int per = (nsets + 1023) / 1024;
  const int b = min(nsets, t * per), e = min(nsets, b + per);
  int sum = 0;
  for (int s = b; s < e; ++s) sum += (off[s + 1] - off[s] + ch - 1) / ch;
  part[t] = sum;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {  // inclusive scan
    const int v = t >= d ? part[t - d] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int acc = part[t] - sum;
  for (int s = b; s < e; ++s) {
    chunk0[s] = acc;
    acc += (off[s + 1] - off[s] + ch - 1) / ch;
  }
  if (t == 1023) chunk0[nsets] = part[1023];
}

// Workgroup g builds chunk g of all sets' chunks (its set by binary search).
template <unsigned OUT>
__global__ __launch_bounds__((Rec32<OUT, true, true>::kChunk)) void row32_set_records_kernel(
    Row32Batch b, const Src8* __restrict__ src) {
  using R = Rec32<OUT, true, true>;
  const int g = blockIdx.x;
  if (g >= b.chunk0[b.nsets]) return;  // uniform over the workgroup
  int lo = 0, hi = b.nsets - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (b.chunk0[mid] <= g) lo = mid;
    else hi = mid - 1;
  }
  const int off = b.set_off[lo];
  const int64_t c0 = b.chunk0[lo];
  row32_records<OUT, true, true>(src + off, b.set_off[lo + 1] - off, g - static_cast<int>(c0),
                           b.rec + c0 * R::kChunk * R::kStride, b.box + c0 * kBox32);
}

// Adds the splits of a row in order and stores.  grid (items * rows_per_item)
template <unsigned OUT>
__global__ __launch_bounds__(kRow) void row32_batch_reduce_kernel(FusedArgs a, Row32Batch b,
                                                                  int splits) {
  using S = Slots<OUT>;
  const int w = static_cast<int>(blockIdx.x);
  Row32Item it;
  if (!row32_item(b, w, &it)) return;
  const int kt = it.row * kRow + static_cast<int>(threadIdx.x);
  double ens = 0.0;
  if (kt < it.n) {
    const int64_t k = static_cast<int64_t>(it.off) + kt;
    double T[kNAcc], G[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < kNAcc; ++q) T[q] = 0.0;
    for (int sp = 0; sp < splits; ++sp) {
      const double* P = a.part + static_cast<int64_t>(sp) * S::nslot * a.pld;
#pragma unroll
      for (int q = 0; q < kNAcc; ++q)
        if (S::used(q)) T[q] += P[S::packed(q) * a.pld + k];
#pragma unroll
      for (int c = 0; c < 3; ++c) G[c] += P[(S::nacc + c) * a.pld + k];
    }
    ens = store_target<OUT, true>(a, a.src[k], a.perm[k], T, G, 1.0 / a.src[it.off].s);
  }
  if constexpr (S::ens) {
    ens = wave_sum(ens);
    if (threadIdx.x == 0) a.ens_part[w] = ens;
  }
}

int nslots(unsigned mask) {
  int c = 0;
  for (unsigned b = 1; b <= VPM_OUT_ENSTROPHY; b <<= 1) c += (mask & b) ? 3 : 0;
  return c + ((mask & VPM_OUT_STRETCH) ? 3 : 0);
}

// Source splits.  Rows that sum in FP64 on every chunk read 88 bytes per
// source, the FP64 strengths among them, and the workgroups in flight drift
// apart: more than 16,384 sources do not stay in an XCD's L2, and the rows of a
// ring then wait for it.  Such sets are split that far while the partials
// stay below 512 MB.  Ring with per-particle radii, all five outputs: 98,304
// particles 21.2 -> 17.3 ms, 131,072 34.7 -> 30.1 (tiled 19.5 and 32.1), 262,144
// 146 -> 117 (121); velocity + stretching 11.6 -> 9.5, 17.8 -> 16.6, 71.9 -> 64.8;
// clouds within 5% either way.
constexpr int64_t kL2Sources = 16384;
constexpr size_t kMaxPartials = size_t(512) << 20;

int row32_splits(int64_t n, unsigned mask, bool unif) {
  const int64_t rows = row_count(n);
  const int k = row_splits(rows, n);
  if (!(mask & VPM_OUT_STRETCH) || (unif && mask != VPM_OUT_STRETCH)) return k;
  const size_t per = static_cast<size_t>(nslots(mask)) * rows * kRow * sizeof(double);
  const int64_t fit = std::min<int64_t>(ceil_div(n, kL2Sources), kMaxPartials / per);
  return std::max(k, static_cast<int>(fit));
}

template <unsigned OUT, bool UNIF>
int launch(FusedArgs a, float* rec, double* box, hipStream_t st, int* nblocks) {
  using R = Rec32<OUT, UNIF>;
  const int rows = static_cast<int>(ceil_div(a.n, kRow));
  const int chunks = static_cast<int>(ceil_div(a.n, R::kChunk));
  const size_t per = static_cast<size_t>(Slots<OUT>::nslot) * rows * kRow * sizeof(double);
  int k = std::min(row32_splits(a.n, OUT, UNIF), std::max(1, chunks / kRowWaves));
  if (a.max_splits > 0) k = std::min(k, a.max_splits);
  if (!a.part || a.part_cap / per < 2) k = 1;
  else k = static_cast<int>(std::min<size_t>(k, a.part_cap / per));
  if (k == 1) a.part = nullptr;
  a.pld = static_cast<int64_t>(rows) * kRow;
  hipLaunchKernelGGL((row32_records_kernel<OUT, UNIF>), dim3(chunks), dim3(R::kChunk), 0, st,
                     a.src, a.n, rec, box);
  VPM_LAUNCH_CHECK("row32_records_kernel");
  hipLaunchKernelGGL((row32_kernel<OUT, UNIF, false>), dim3(rows, k), dim3(kRowBlock), 0, st, a,
                     Row32Batch{}, k, rec, box);
  VPM_LAUNCH_CHECK("row32_kernel");
  *nblocks = rows;
  if (k > 1) {
    const int rb = static_cast<int>(ceil_div(a.n, 256));
    hipLaunchKernelGGL((split_reduce_kernel<OUT, UNIF>), dim3(rb), dim3(256), 0, st, a, k);
    VPM_LAUNCH_CHECK("split_reduce_kernel");
    *nblocks = rb;
  }
  return VPM_OK;
}

template <unsigned OUT>
int launch_batch(FusedArgs a, const Row32Batch& b, hipStream_t st) {
  using R = Rec32<OUT, true, true>;
  const int64_t groups = static_cast<int64_t>(b.n_items) * b.rows_per_item;
  if (groups == 0 || a.n == 0) return VPM_OK;
  const int k = a.part ? b.splits : 1;
  if (k == 1) a.part = nullptr;
  a.pld = a.n;
  hipLaunchKernelGGL(row32_chunks_kernel, dim3(1), dim3(1024), 0, st, b.set_off, b.nsets,
                     R::kChunk, b.chunk0);
  VPM_LAUNCH_CHECK("row32_chunks_kernel");
  const int64_t chunks = ceil_div(a.n, R::kChunk) + b.nsets;  // bound; extra groups leave
  hipLaunchKernelGGL(row32_set_records_kernel<OUT>, dim3(static_cast<unsigned>(chunks)),
                     dim3(R::kChunk), 0, st, b, a.src);
  VPM_LAUNCH_CHECK("row32_set_records_kernel");
  hipLaunchKernelGGL((row32_kernel<OUT, true, true>), dim3(static_cast<unsigned>(groups), k),
                     dim3(kRowBlock), 0, st, a, b, k, nullptr, nullptr);
  VPM_LAUNCH_CHECK("row32_kernel");
  if (k > 1) {
    hipLaunchKernelGGL(row32_batch_reduce_kernel<OUT>, dim3(static_cast<unsigned>(groups)),
                       dim3(kRow), 0, st, a, b, k);
    VPM_LAUNCH_CHECK("row32_batch_reduce_kernel");
  }
  return VPM_OK;
}

}  // namespace

// Records of whole chunks, and one group read ahead past the last.
size_t row32_record_bytes(int64_t n) {
  return (static_cast<size_t>(ceil_div(n > 0 ? n : 1, kMaxChunk32)) * kMaxChunk32 + kMaxGroup32) *
         kStride32 * sizeof(float);
}

size_t row32_box_bytes(int64_t n) {
  return static_cast<size_t>(ceil_div(n > 0 ? n : 1, kMinChunk32)) * kBox32 * sizeof(double);
}

size_t row32_split_bytes(int64_t n, unsigned mask, bool unif) {
  const int64_t rows = row_count(n);
  const int k = row32_splits(n, mask, unif);
  return k > 1 ? static_cast<size_t>(k) * nslots(mask) * rows * kRow * sizeof(double) : 0;
}

int row32_run(const FusedArgs& a, unsigned mask, bool unif, float* rec, double* box,
              hipStream_t st, int* nblocks) {
  switch (mask | (unif ? 32u : 0u)) {
#define VPM_ROW32(M, U)      \
  case (M) | ((U) ? 32u : 0u): \
    return launch<M, U>(a, rec, box, st, nblocks);
    VPM_ROW32(1u, true) VPM_ROW32(2u, true) VPM_ROW32(3u, true) VPM_ROW32(4u, true)
    VPM_ROW32(7u, true) VPM_ROW32(8u, true) VPM_ROW32(16u, true) VPM_ROW32(24u, true)
    VPM_ROW32(26u, true) VPM_ROW32(27u, true) VPM_ROW32(31u, true)
    VPM_ROW32(1u, false) VPM_ROW32(2u, false) VPM_ROW32(3u, false) VPM_ROW32(4u, false)
    VPM_ROW32(7u, false) VPM_ROW32(8u, false) VPM_ROW32(16u, false) VPM_ROW32(24u, false)
    VPM_ROW32(26u, false) VPM_ROW32(27u, false) VPM_ROW32(31u, false)
#undef VPM_ROW32
    default:
      return fail(VPM_ERR_ARG, "row32: unknown output set");
  }
}

int row32_batch_splits(int64_t n, int n_items, int rows_per_item) {
  // Rows of equal sets run in rounds of 768 workgroups; unequal ones, largest
  // first, need a few rounds' worth to end together.
  const int64_t rows = std::min<int64_t>(static_cast<int64_t>(n_items) * rows_per_item,
                                         ceil_div(n, kRow) + n_items);
  return static_cast<int>(std::clamp<int64_t>(3 * 768 / std::max<int64_t>(rows, 1), 1, 8));
}

size_t row32_batch_split_bytes(int64_t n, int splits) {
  return splits > 1 ? static_cast<size_t>(splits) * nslots(31u) * n * sizeof(double) : 0;
}

size_t row32_batch_record_bytes(int64_t n, int nsets) {
  return (static_cast<size_t>(n) + static_cast<size_t>(kMaxChunk32) * nsets + kMaxGroup32) *
         kStride32 * sizeof(float);
}

size_t row32_batch_box_bytes(int64_t n, int nsets) {
  return (static_cast<size_t>(n) / kMinChunk32 + nsets + 1) * kBox32 * sizeof(double);
}

int row32_batch_run(const FusedArgs& a, const Row32Batch& b, unsigned mask, hipStream_t st) {
  switch (mask) {
    case 3u: return launch_batch<3u>(a, b, st);
    case 7u: return launch_batch<7u>(a, b, st);
    case 27u: return launch_batch<27u>(a, b, st);
    default: return launch_batch<31u>(a, b, st);
  }
}

}  // namespace vpm
