// What the kernels of the fused FP32-compensated pass share: arguments, the
// accumulator slots, the FP64 epilogue, the coherence test and the reduction
// of source splits.
#pragma once

#include "vpm_common.h"

namespace vpm {

struct FusedArgs {
  int n;
  const Src8* src;      // sorted particles
  const int* perm;      // sorted k -> caller index (null: identity)
  double* vel;          // outputs (caller order); unrequested ones point to scratch
  double* str;
  double* pse;
  double* vort;
  int64_t ld_vel, ld_str, ld_pse, ld_vort;
  double* ens_part;     // per-block enstrophy partials
  // Source split: workgroup (b, k) sums sources [k*chunk, (k+1)*chunk) into
  // part + k*nslot*pld (FP64 raw sums per target, by sorted index); a reduce
  // kernel adds the splits in order k = 0, 1, ... and stores.  part == null:
  // one split, stored directly.
  double* part;
  size_t part_cap;      // bytes available at part
  int max_splits;       // 0: automatic
  int g64_mode;         // VPM_G64_*: per-pair FP64 alpha_j sum of the stretching
  int64_t pld;
  int chunk;
  // Far-field records of the FP32 pass (far_records_kernel): per chunk of
  // SUB sorted sources its centre and half-extent in radius units (far_box, 6 doubles)
  // and per source FP32 chunk-centred offsets, strength and moment
  // (far_rec, FarRec<OUT>::kStride floats).  Null where unused.
  const float* far_rec;
  const double* far_box;
};

namespace {

// Accumulator slots; kH is the moment sum of the far-field form (folded into
// kU's FP64 totals per sub-tile, never stored).
// kT9 is the far-field form's sum of the PSE weights (folded into kP's
// partials per sub-tile, never stored).
enum : int { kU = 0, kG = 3, kSd = 6, kP = 9, kW = 12, kE = 15, kH = 18, kT9 = 21, kNAcc = 22 };

template <unsigned OUT>
struct Slots {
  static constexpr bool vel = OUT & VPM_OUT_VEL, str = OUT & VPM_OUT_STRETCH,
                        pse = OUT & VPM_OUT_PSE, vort = OUT & VPM_OUT_VORT,
                        ens = OUT & VPM_OUT_ENSTROPHY;
  // Slots with FP64 totals.  The stretching's alpha_j sum G has FP64
  // totals of its own (gsum): waves whose targets' strengths are coherent
  // (vortex rings, tubes, sheets) add to it in FP64 per pair on near tiles,
  // because there alpha_i x G is a near-exact cancellation and FP32 partials
  // of G cost an order of magnitude in the stretching's relative error
  // (coherent_wave below); other waves, and every wave on far tiles, fold
  // FP32 partials kG..kG+2 into it per sub-tile.
  static __host__ __device__ constexpr bool used(int k) {
    return (k < 3 && vel) || (k >= 6 && k < 9 && str) || (k >= 9 && k < 12 && pse) ||
           (k >= 12 && k < 15 && vort) || (k >= 15 && k < 18 && ens);
  }
  // position of slot k among the used ones (the split partial layout)
  static __host__ __device__ constexpr int packed(int k) {
    int c = 0;
    for (int q = 0; q < k; ++q) c += used(q) ? 1 : 0;
    return c;
  }
  static constexpr int nacc = packed(kNAcc);
  static constexpr int nslot = nacc + (str ? 3 : 0);  // + the FP64 alpha_j sum
};

// Scaling and storing of one target's totals T (FP32-pass slots, FP64) and G
// (the FP64 alpha_j sum of the stretching); returns its enstrophy term.
template <unsigned OUT, bool UNIF>
__device__ __forceinline__ double store_target(const FusedArgs& a, const Src8& ti, int64_t o,
                                               const double* T, const double* G, double scale) {
  using S = Slots<OUT>;
  const double C = kOneOverFourPi;
  double s1 = 1.0, s2 = 1.0, s3 = 1.0;  // 1/sigma^k for uniform sigma
  if constexpr (UNIF) {
    s1 = scale;
    s2 = scale * scale;
    s3 = s2 * scale;
  }
  if constexpr (S::vel) {
    const double f = -C * s2;
    a.vel[o] = f * T[kU + 0];
    a.vel[a.ld_vel + o] = f * T[kU + 1];
    a.vel[2 * a.ld_vel + o] = f * T[kU + 2];
  }
  if constexpr (S::str) {
    const double ax = ti.ax, ay = ti.ay, az = ti.az;
    const double f = C * s3;
    a.str[o] = f * ((ay * G[2] - az * G[1]) + T[kSd + 0]);
    a.str[a.ld_str + o] = f * ((az * G[0] - ax * G[2]) + T[kSd + 1]);
    a.str[2 * a.ld_str + o] = f * ((ax * G[1] - ay * G[0]) + T[kSd + 2]);
  }
  if constexpr (S::pse) {
    const double f = 105.0 * ti.nu * C * s2;
    a.pse[o] = f * T[kP + 0];
    a.pse[a.ld_pse + o] = f * T[kP + 1];
    a.pse[2 * a.ld_pse + o] = f * T[kP + 2];
  }
  if constexpr (S::vort) {
    const double f = 7.5 * C * s3;
    a.vort[o] = f * T[kW + 0];
    a.vort[a.ld_vort + o] = f * T[kW + 1];
    a.vort[2 * a.ld_vort + o] = f * T[kW + 2];
  }
  if constexpr (S::ens) return (ti.ax * T[kE + 0] + ti.ay * T[kE + 1] + ti.az * T[kE + 2]) * s1;
  return 0.0;
}

// Non-inline constants of the pair update, held in registers by the caller:
// as literal operands (v_fmac_f32 v, 0x3fc00000, v) they halve the issue rate
// of their instruction on gfx950.
template <typename Real>
struct PairConst {
  Real c15, c75, c22, c3, c25;
  Real c45;  // the row pass with per-particle radii
};

// Constant-address-space view of the records: a load through it with a
// wave-uniform address becomes a scalar (s_load) load.
typedef __attribute__((address_space(4))) const float far_float_t;

// Coherence of 64 consecutive sorted targets (one lane row of a wave),
// |sum alpha_i| / sum |alpha_i|: for unrelated strengths it is ~0.14 and
// stayed below 0.35 over the 16384 rows of a random cloud of 2^20 particles;
// along vortex rings, tubes and sheets (the example cases, leapfrogging
// rings) it stayed above 0.59.  A wave with a row above kCoherent sums G in
// FP64 per pair.
constexpr double kCoherent = 0.45;

template <int R>
__device__ __forceinline__ bool coherent_wave(const Src8* tg, const bool* valid) {
  bool any = false;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    double sx = 0.0, sy = 0.0, sz = 0.0, m = 0.0;
    if (valid[r]) {
      sx = tg[r].ax;
      sy = tg[r].ay;
      sz = tg[r].az;
      m = sqrt(sx * sx + sy * sy + sz * sz);
    }
    sx = wave_sum(sx);
    sy = wave_sum(sy);
    sz = wave_sum(sz);
    m = wave_sum(m);
    any = any || sqrt(sx * sx + sy * sy + sz * sz) > kCoherent * m;
  }
  return any;
}

// Adds the splits' raw sums in split order (deterministic) and stores; one
// enstrophy partial per workgroup.
template <unsigned OUT, bool UNIF>
__global__ __launch_bounds__(256) void split_reduce_kernel(FusedArgs a, int nsplit) {
  using S = Slots<OUT>;
  __shared__ double red[4];
  const int k = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  double ens_local = 0.0;
  if (k < a.n) {
    double T[kNAcc], G[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < kNAcc; ++q) T[q] = 0.0;
    for (int sp = 0; sp < nsplit; ++sp) {
      const double* P = a.part + static_cast<int64_t>(sp) * S::nslot * a.pld;
#pragma unroll
      for (int q = 0; q < kNAcc; ++q)
        if (S::used(q)) T[q] += P[S::packed(q) * a.pld + k];
      if constexpr (S::str) {
#pragma unroll
        for (int c = 0; c < 3; ++c) G[c] += P[(S::nacc + c) * a.pld + k];
      }
    }
    const double scale = UNIF ? 1.0 / a.src[0].s : 1.0;
    ens_local = store_target<OUT, UNIF>(a, a.src[k], a.perm ? a.perm[k] : k, T, G, scale);
  }
  if constexpr (S::ens) {
    const double bs = block_sum<256>(ens_local, red);
    if (threadIdx.x == 0) a.ens_part[blockIdx.x] = bs;
  }
}

}  // namespace

}  // namespace vpm
