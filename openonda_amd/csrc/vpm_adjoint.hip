// Hand-written adjoint (vector-Jacobian product) of the fused pair pass.
//
// Given cotangents lam (of the self-induced velocity u), mu (of the
// stretching S) and xi (of the PSE term D), computes dL/dx and dL/dalpha for
// L = sum_k lam_k.u_k + mu_k.S_k + xi_k.D_k with the GPU-plugin arithmetic
// (sigma_ij, nu_i; ParticlesPhysicsCuda.py:159-191, :396-440, :500-525) and
// sigma held fixed.  One symmetric all-pairs pass per particle m accumulates
// both of its roles -- m as target and m as source -- from its partners' data
// staged in LDS, so no atomics and no second pass are needed.
//
// With r = x_m - x_j, rho^2 = r^2/s^2, t = (rho^2+1)^-1/2, s = sigma_ij, and
//   g = (rho^2+2.5) t^5/s^3,  f = 3(rho^2+3.5) t^7/s^5 = -2 dg/dr^2,
//   h = 7.5(rho^2+4.5) t^9/s^7 = -df/dr^2,  p = t^9/s^2,  q = 4.5 t^11/s^4 = -dp/dr^2,
//   c = r x a_j,  d_mu = mu_m - mu_j,  Q_j = a_j x mu_j,  P_m = a_m x mu_m,
//   phi = d_mu.r,  psi = a_m.c,  z = nu xi,  C = 1/(4 pi):
// velocity  dA_m += C g (lam_j x r)
//           dX_m += C f [lam_m.c - a_m.(lam_j x r)] r - C g [a_j x lam_m - a_m x lam_j]
// stretch   dA_m += C [g (a_j x d_mu) + f phi c]
//           dX_m += C [(f (a_j.P_m + a_m.Q_j) - 2 h psi phi) r + f phi (a_j x a_m) + f psi d_mu]
// PSE       dA_m += 105 C p (z_j - z_m)
//           dX_m += -2 * 105 C q ((a_j - a_m).(z_m - z_j)) r
// Sums over j of g a_j, g lam_j and f phi a_j are accumulated per target and
// crossed with the target's vectors once; the three radial terms share one
// accumulator.
// Precision F32C runs the rows of vpm_adj32.hip above kAdjRowsMax particles,
// F64 and smaller sets the FP64 rows here.

#include <algorithm>
#include <type_traits>

#include "vpm_adj32.h"
#include "vpm_common.h"
#include "vpm_prepass.h"
#include "vpm_rows.h"

namespace vpm {

namespace {

// ---- FP64 rows (vpm_rows.h): any subset of the cotangents, sigma_ij ------
// The lengths are not scaled: sc = 1 in the formulas above.  Per pair
//   k = lam_j x r - Q_j,  E = lam_m.c - a_m.k + a_j.P_m,
// G = sum g a_j, Lam = sum g lam_j, A = sum g k + 105 p (z_j - z_m),
// B = sum f phi c, X = sum [f E - 2 h psi phi + 945 q (a_j - a_m).(z_j - z_m)] r,
// Y = sum f phi a_j, D = sum f psi (mu_m - mu_j); then
//   dA = C (A + G x mu_m + B),  dX = C (X - G x lam_m + a_m x Lam + Y x a_m + D).
// The pair j = m is left out: its terms cancel or vanish.
//
// Bound by FP64 issue (about 95 instructions per pair with all three
// cotangents).  One rsq64 per pair in place of an IEEE square root and
// division, the sums G, Lam, Y, D crossed once per particle, the sources as
// scalar operands and rows of 64 in place of blocks of 256: all cotangents,
// general radius, 1,000 particles 483 -> 29 us, 10,007 825 -> 369 us, 50,021
// 13.7 -> 8.0 ms.

// Record of one particle, in the caller's order: x 0, a 3, lam 6, mu 9,
// z = nu xi 12, Q = a x mu 15, sigma 18.
constexpr int kRec64 = 20;

__global__ __launch_bounds__(256) void adj64_records_kernel(vpm_particles_t p,
                                                            const double* __restrict__ lam,
                                                            const double* __restrict__ mu,
                                                            const double* __restrict__ xi,
                                                            int64_t ldc, double* __restrict__ rec) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= p.n) return;
  double* r = rec + i * kRec64;
  const double nu = xi ? p.nu[i] : 0.0;
  double a[3], m[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    a[c] = p.str[c * p.ld + i];
    m[c] = mu ? mu[c * ldc + i] : 0.0;
    r[c] = p.pos[c * p.ld + i];
    r[3 + c] = a[c];
    r[6 + c] = lam ? lam[c * ldc + i] : 0.0;
    r[9 + c] = m[c];
    r[12 + c] = xi ? nu * xi[c * ldc + i] : 0.0;
  }
  r[15] = a[1] * m[2] - a[2] * m[1];
  r[16] = a[2] * m[0] - a[0] * m[2];
  r[17] = a[0] * m[1] - a[1] * m[0];
  r[18] = p.sigma[i];
  r[19] = 0.0;
}

struct Adj64Acc {
  double G[3], L[3], A[3], B[3], X[3], Y[3], D[3];
};

__device__ __forceinline__ double dot3(const double* a, const double* b, double c) {
  return ::fma(a[2], b[2], ::fma(a[1], b[1], ::fma(a[0], b[0], c)));
}
__device__ __forceinline__ void add3(double* s, double w, const double* v) {
  s[0] = ::fma(w, v[0], s[0]);
  s[1] = ::fma(w, v[1], s[1]);
  s[2] = ::fma(w, v[2], s[2]);
}
__device__ __forceinline__ void add_cross(double* o, const double* a, const double* b) {
  o[0] = ::fma(-a[2], b[1], ::fma(a[1], b[2], o[0]));
  o[1] = ::fma(-a[0], b[2], ::fma(a[2], b[0], o[1]));
  o[2] = ::fma(-a[1], b[0], ::fma(a[0], b[1], o[2]));
}

// t: the target's record (half its radius at 18), s: the source's.
template <unsigned OUT>
__device__ __forceinline__ void adj64_pair(Adj64Acc& acc, const double* t, const double* s) {
  constexpr bool vel = OUT & VPM_OUT_VEL, str = OUT & VPM_OUT_STRETCH, pse = OUT & VPM_OUT_PSE;
  const double d[3] = {t[0] - s[0], t[1] - s[1], t[2] - s[2]};
  const double sg = ::fma(0.5, s[18], t[18]);
  const double s2 = sg * sg;
  const double D = dot3(d, d, s2);
  const double t1 = (vel || str) ? rsq64(D) : rsq64_inf(D);
  const double t2 = t1 * t1, t3 = t2 * t1, w = s2 * t2;
  const double *a = s + 3, *l = s + 6, *m = s + 9, *z = s + 12, *Q = s + 15;
  double xc = 0.0;
  if constexpr (vel || str) {
    const double t5 = t3 * t2;
    const double g = t3 * ::fma(1.5, w, 1.0);
    const double f = t5 * ::fma(7.5, w, 3.0);
    const double c[3] = {d[1] * a[2] - d[2] * a[1], d[2] * a[0] - d[0] * a[2],
                         d[0] * a[1] - d[1] * a[0]};
    double k[3] = {0.0, 0.0, 0.0}, E = 0.0;
    add3(acc.G, g, a);
    if constexpr (vel) {
      k[0] = l[1] * d[2] - l[2] * d[1];
      k[1] = l[2] * d[0] - l[0] * d[2];
      k[2] = l[0] * d[1] - l[1] * d[0];
      add3(acc.L, g, l);
      E = dot3(t + 6, c, 0.0);
    }
    if constexpr (str) {
      k[0] -= Q[0];
      k[1] -= Q[1];
      k[2] -= Q[2];
      E = dot3(t + 15, a, E);
    }
    add3(acc.A, g, k);
    xc = f * (E - dot3(t + 3, k, 0.0));
    if constexpr (str) {
      const double dm[3] = {t[9] - m[0], t[10] - m[1], t[11] - m[2]};
      const double phi = dot3(dm, d, 0.0), psi = dot3(t + 3, c, 0.0);
      const double fphi = f * phi;
      add3(acc.B, fphi, c);
      add3(acc.Y, fphi, a);
      add3(acc.D, f * psi, dm);
      const double h = (t5 * t2) * ::fma(-52.5, w, -15.0);  // -2 h
      xc = ::fma(h * psi, phi, xc);
    }
  }
  if constexpr (pse) {
    const double p = (sg * t3) * (w * w * w);
    const double dz[3] = {z[0] - t[12], z[1] - t[13], z[2] - t[14]};
    const double da[3] = {a[0] - t[3], a[1] - t[4], a[2] - t[5]};
    add3(acc.A, 105.0 * p, dz);
    xc = ::fma(945.0 * (p * t2), dot3(da, dz, 0.0), xc);
  }
  add3(acc.X, xc, d);
}

// grid (rows, splits); components 0..2 dL/dx, 3..5 dL/dalpha.
template <unsigned OUT>
__global__ __launch_bounds__(kRowBlock, 4) void adj64_kernel(RowArgs A,
                                                             const double* __restrict__ rec) {
  __shared__ double red[kRowWaves][6][kRow];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kRow;
  const int64_t i = row0 + lane;
  double t[19];
  {
    const double* r = rec + (i < A.m ? i : row0) * kRec64;
#pragma unroll
    for (int q = 0; q < 19; ++q) t[q] = r[q];
    t[18] *= 0.5;
  }
  int64_t b, e;
  row_share(0, A.n, static_cast<int>(blockIdx.y) * kRowWaves + wave, A.splits * kRowWaves, &b, &e);
  const int64_t o0 = row0 < b ? b : (row0 < e ? row0 : e);
  const int64_t o1 = row0 + kRow < b ? b : (row0 + kRow < e ? row0 + kRow : e);
  Adj64Acc acc{};
  auto load = [&](double* s, int64_t j) {
    const scalar_double_t* r = (const scalar_double_t*)(rec + j * kRec64);
#pragma unroll
    for (int q = 0; q < 19; ++q) s[q] = r[q];
  };
  for (int64_t j = o0; j < o1; ++j) {
    double s[19];
    load(s, j);
    if (j != i) adj64_pair<OUT>(acc, t, s);
  }
#pragma unroll 1
  for (int side = 0; side < 2; ++side) {
    const int64_t j1 = side ? e : o0;
    for (int64_t j = side ? o1 : b; j < j1; ++j) {
      double s[19];
      load(s, j);
      adj64_pair<OUT>(acc, t, s);
    }
  }
  {
    constexpr bool vel = OUT & VPM_OUT_VEL, str = OUT & VPM_OUT_STRETCH;
    double v[6] = {acc.X[0], acc.X[1], acc.X[2], acc.A[0], acc.A[1], acc.A[2]};
    if constexpr (vel) {
      add_cross(v, t + 6, acc.G);
      add_cross(v, t + 3, acc.L);
    }
    if constexpr (str) {
      add_cross(v, acc.Y, t + 3);
      add_cross(v + 3, acc.G, t + 9);
      for (int q = 0; q < 3; ++q) {
        v[q] += acc.D[q];
        v[3 + q] += acc.B[q];
      }
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) red[wave][q][lane] = kOneOverFourPi * v[q];
  }
  __syncthreads();
  if (wave >= 6) return;
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) s += red[w][wave][lane];
  if (A.part) {
    const int64_t pm = static_cast<int64_t>(gridDim.x) * kRow;
    A.part[(static_cast<int64_t>(blockIdx.y) * 6 + wave) * pm + i] = s;
  } else if (i < A.m) {
    A.out[wave / 3][(wave % 3) * A.ld_out + i] = s;
  }
}

template <unsigned OUT>
int launch_adj64(RowArgs a, const double* rec, void* part, size_t part_bytes, int max_splits,
                 hipStream_t st) {
  const int64_t rows = row_count(a.m);
  const size_t per = row_split_bytes(rows, 6, false);
  int k = row_splits(rows, a.n);
  if (max_splits > 0) k = std::min(k, max_splits);
  k = part ? static_cast<int>(std::max<size_t>(1, std::min<size_t>(k, part_bytes / per))) : 1;
  a.splits = k;
  a.part = k > 1 ? static_cast<double*>(part) : nullptr;
  hipLaunchKernelGGL(adj64_kernel<OUT>, dim3(static_cast<unsigned>(rows), k), dim3(kRowBlock), 0,
                     st, a, rec);
  VPM_LAUNCH_CHECK("adj64_kernel");
  if (k > 1) {
    hipLaunchKernelGGL(row_reduce_kernel, dim3(static_cast<unsigned>(ceil_div(a.m, 256)), 6),
                       dim3(256), 0, st, a, 6, rows * kRow);
    VPM_LAUNCH_CHECK("row_reduce_kernel");
  }
  return VPM_OK;
}

int adj64_run(const RowArgs& a, unsigned mask, const double* rec, void* part, size_t part_bytes,
              int max_splits, hipStream_t st) {
  switch (mask) {
    case 1u: return launch_adj64<1u>(a, rec, part, part_bytes, max_splits, st);
    case 2u: return launch_adj64<2u>(a, rec, part, part_bytes, max_splits, st);
    case 3u: return launch_adj64<3u>(a, rec, part, part_bytes, max_splits, st);
    case 4u: return launch_adj64<4u>(a, rec, part, part_bytes, max_splits, st);
    case 5u: return launch_adj64<5u>(a, rec, part, part_bytes, max_splits, st);
    case 6u: return launch_adj64<6u>(a, rec, part, part_bytes, max_splits, st);
    default: return launch_adj64<7u>(a, rec, part, part_bytes, max_splits, st);
  }
}

// Sets up to this size run the FP64 rows also in the FP32-compensated
// precision: the FP32 rows are twice as fast per pair, but first sort and
// write records.  FP64 / FP32 rows, cloud, uniform radius: all three
// cotangents, 1,000 particles 28 / 54 us, 4,000 73 / 86, 5,000 107 / 106,
// 6,000 145 / 120; velocity and stretching only 5,000 90 / 92, 6,000 122 /
// 104; velocity only 5,000 65 / 67, 6,000 88 / 74.
constexpr int64_t kAdjRowsMax = 5120;

bool adj_rows_wanted(int64_t n, const vpm_forward_opts_t* o) {
  return o->precision == VPM_PREC_F64 || n <= kAdjRowsMax;
}

struct AdjLayout {
  size_t bbox_part, bbox, keys_in, keys_out, idx_in, perm, rec, box, split, cub, total, cub_bytes,
      split_bytes;
};

// rec: the FP64 rows' records, or those of the FP32 rows.
int adj_layout(int64_t n, const vpm_forward_opts_t* o, AdjLayout* L) {
  const bool rows = adj_rows_wanted(n, o);
  const size_t N = static_cast<size_t>(n > 0 ? n : 1);
  size_t off = 0;
  auto take = [&](size_t b) {
    const size_t at = off;
    off += align256(b);
    return at;
  };
  L->bbox_part = take(kBboxBlocks * 6 * sizeof(double));
  L->bbox = take(8 * sizeof(double));
  L->keys_in = take((N + kSamples) * 4);
  L->keys_out = take(N * 4);
  L->idx_in = take(N * 4);
  L->perm = take(N * 4);
  L->rec = take(rows ? N * kRec64 * sizeof(double) : adj32_record_bytes(n));
  L->box = take(rows ? 0 : adj32_box_bytes(n));
  L->split_bytes = rows ? row_workspace_bytes(n, n, 6) : adj32_split_bytes(n);
  L->split = take(L->split_bytes);
  size_t cb = 0;
  if (!rows && !o->presorted) {
    const int rc = sort_temp_bytes(n, &cb);
    if (rc) return rc;
  }
  L->cub_bytes = cb;
  L->cub = take(cb + 16);
  L->total = off;
  return VPM_OK;
}

// ---- velocity at evaluation points: adjoint w.r.t. the sources (FP64) ----
// For u(y_i) = -C sum_j g_ij (r_ij x a_j), r_ij = y_i - x_j, sigma_j,
// r^2 > 1e-8 (ParticlesPhysicsCuda.py:65-97):
//   dA_j = C sum_i g (r x lam_i),  dX_j = C sum_i [g (a_j x lam_i) - f (r.(a_j x lam_i)) r].
// The particles are the rows' targets and the points the sources (vpm_rows.h):
// with r' = x_j - y_i = -r and c = r' x lam_i, dA_j = -C sum g c and
// dX_j = C [a_j x sum g lam_i + sum f (a_j . c) r'].  The radius is the
// target's, so its square enters the factors as constants: t^3 (1 + 1.5 w) =
// t^3 + (1.5 s^2) t^5.  Bound: FP64 issue, 38 instructions per pair (4,096
// points, 131,072 particles: 765 us; 794 us with w = s^2 t^2 formed per pair;
// 1820 us with the points staged in LDS, IEEE root and division, and a_j x
// lam_i per pair).
struct OpVelAtAdjoint {
  static constexpr bool kTargetData = true, kRadius = false, kNu = false, kSkipSelf = false;
  static constexpr int kOut = 6;
  static constexpr bool kSum = false, kSelfTerm = false;
  struct Acc { double A[3] = {0, 0, 0}, L[3] = {0, 0, 0}, X[3] = {0, 0, 0}; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = ::fma(rx, rx, ::fma(ry, ry, rz * rz));
    if (r2 > kEpsPair) {
      const double s2 = t.s * t.s;
      const double tt = rsq64(r2 + s2);
      const double t2 = tt * tt, t3 = t2 * tt, t5 = t3 * t2;
      const double g = ::fma(1.5 * s2, t5, t3);
      const double cx = ry * s.az - rz * s.ay;
      const double cy = rz * s.ax - rx * s.az;
      const double cz = rx * s.ay - ry * s.ax;
      const double e = t5 * ::fma(7.5 * s2, t2, 3.0) *
                       ::fma(t.ax, cx, ::fma(t.ay, cy, t.az * cz));
      a.A[0] = ::fma(-g, cx, a.A[0]);
      a.A[1] = ::fma(-g, cy, a.A[1]);
      a.A[2] = ::fma(-g, cz, a.A[2]);
      a.L[0] = ::fma(g, s.ax, a.L[0]);
      a.L[1] = ::fma(g, s.ay, a.L[1]);
      a.L[2] = ::fma(g, s.az, a.L[2]);
      a.X[0] = ::fma(e, rx, a.X[0]);
      a.X[1] = ::fma(e, ry, a.X[1]);
      a.X[2] = ::fma(e, rz, a.X[2]);
    }
  }
  // components 0..2: dL/dx, 3..5: dL/dalpha
  static __device__ inline void result(const Acc& a, const RowTarget& t, double* v) {
    v[0] = kOneOverFourPi * ((t.ay * a.L[2] - t.az * a.L[1]) + a.X[0]);
    v[1] = kOneOverFourPi * ((t.az * a.L[0] - t.ax * a.L[2]) + a.X[1]);
    v[2] = kOneOverFourPi * ((t.ax * a.L[1] - t.ay * a.L[0]) + a.X[2]);
    for (int c = 0; c < 3; ++c) v[3 + c] = kOneOverFourPi * a.A[c];
  }
};

int vel_at_adjoint(const vpm_points_t* targets, const vpm_particles_t* src, const double* lam,
                   int64_t ld_lam, double* dpos, double* dstr, int64_t ld_out, void* ws,
                   size_t ws_bytes, void* stream, const char* who) {
  int rc = check_points(targets, who);
  if (rc) return rc;
  if ((rc = check_particles(src, false, who))) return rc;
  if (targets->m > 0 && (!lam || ld_lam < targets->m)) {
    set_error("%s: bad cotangent", who);
    return VPM_ERR_ARG;
  }
  if (src->n > 0 && (!dpos || !dstr || ld_out < src->n)) {
    set_error("%s: bad output", who);
    return VPM_ERR_ARG;
  }
  RowArgs a{};
  a.m = src->n;
  a.tpos = src->pos;
  a.tq = src->str;
  a.tld = a.tqld = src->ld;
  a.ts = src->sigma;
  a.n = targets->m;
  a.pos = targets->pos;
  a.ld = targets->ld;
  a.q = lam;
  a.qld = ld_lam;
  a.out[0] = dpos;
  a.out[1] = dstr;
  a.ld_out = ld_out;
  return row_launch<OpVelAtAdjoint>(a, ws, ws_bytes, as_stream(stream), "vel_at_adjoint");
}

}  // namespace

}  // namespace vpm

using namespace vpm;

extern "C" {

// Enough for either precision, so that one workspace serves both.
size_t vpm_adjoint_workspace_bytes(int64_t n, const vpm_forward_opts_t* opts) {
  vpm_forward_opts_t o{};
  o.presorted = opts ? opts->presorted : 0;
  size_t most = 0;
  for (const int precision : {VPM_PREC_F64, VPM_PREC_F32C}) {
    o.precision = precision;
    AdjLayout L{};
    if (adj_layout(n, &o, &L) != VPM_OK) return 0;
    most = std::max(most, L.total);
  }
  return most;
}

int vpm_adjoint(const vpm_particles_t* p, const vpm_adjoint_in_t* in, const vpm_forward_opts_t* o,
                vpm_adjoint_out_t* out, void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  if (!in || !o || !out) return fail(VPM_ERR_ARG, "vpm_adjoint: null argument");
  unsigned mask = 0;
  if (in->lam) mask |= VPM_OUT_VEL;
  if (in->mu) mask |= VPM_OUT_STRETCH;
  if (in->xi) mask |= VPM_OUT_PSE;
  if (o->precision != VPM_PREC_F64 && o->precision != VPM_PREC_F32C)
    return fail(VPM_ERR_ARG, "vpm_adjoint: unknown precision");
  if (o->sigma_mode != VPM_SIGMA_GENERAL && o->sigma_mode != VPM_SIGMA_UNIFORM)
    return fail(VPM_ERR_ARG, "vpm_adjoint: unknown sigma mode");
  int rc = check_particles(p, in->xi != nullptr, "vpm_adjoint");
  if (rc) return rc;
  const int64_t n = p->n;
  if (in->ld < n) return fail(VPM_ERR_ARG, "vpm_adjoint: cotangent ld < n");
  if (out->ld < n || (n && (!out->dpos || !out->dstr)))
    return fail(VPM_ERR_ARG, "vpm_adjoint: bad output");
  AdjLayout L{};
  if ((rc = adj_layout(n, o, &L))) return rc;
  if (!workspace || ws_bytes < L.total) {
    set_error("vpm_adjoint: workspace %zu bytes < required %zu", ws_bytes, L.total);
    return VPM_ERR_WORKSPACE;
  }
  if (n == 0) return VPM_OK;
  if (o->max_splits < 0) return fail(VPM_ERR_ARG, "vpm_adjoint: max_splits < 0");
  if (mask == 0) mask = VPM_OUT_VEL;  // all cotangents null: zero gradients from the vel pass
  hipStream_t st = as_stream(stream);
  char* ws = static_cast<char*>(workspace);
  void* part = L.split_bytes ? ws + L.split : nullptr;
  if (adj_rows_wanted(n, o)) {
    double* rec = reinterpret_cast<double*>(ws + L.rec);
    hipLaunchKernelGGL(adj64_records_kernel, dim3(static_cast<unsigned>(ceil_div(n, 256))),
                       dim3(256), 0, st, *p, in->lam, in->mu, in->xi, in->ld, rec);
    VPM_LAUNCH_CHECK("adj64_records_kernel");
    RowArgs a{};
    a.m = a.n = n;
    a.out[0] = out->dpos;
    a.out[1] = out->dstr;
    a.ld_out = out->ld;
    return adj64_run(a, mask, rec, part, L.split_bytes, o->max_splits, st);
  }
  int* perm = nullptr;
  if (!o->presorted) {
    perm = reinterpret_cast<int*>(ws + L.perm);
    rc = morton_sort(p, reinterpret_cast<double*>(ws + L.bbox_part),
                     reinterpret_cast<double*>(ws + L.bbox), reinterpret_cast<uint32_t*>(ws + L.keys_in),
                     reinterpret_cast<uint32_t*>(ws + L.keys_out), reinterpret_cast<int*>(ws + L.idx_in),
                     perm, ws + L.cub, L.cub_bytes, nullptr, st);
    if (rc) return rc;
  }
  return adj32_run(Adj32Args{*p, in->lam, in->mu, in->xi, in->ld, perm, out->dpos, out->dstr,
                             out->ld, reinterpret_cast<float*>(ws + L.rec),
                             reinterpret_cast<double*>(ws + L.box), static_cast<double*>(part),
                             L.split_bytes, o->max_splits, o->sigma_mode == VPM_SIGMA_UNIFORM},
                   mask, st);
}

int vpm_induced_velocity_at_adjoint(const vpm_points_t* targets, const vpm_particles_t* src,
                                    const double* lam, int64_t ld_lam, double* dpos, double* dstr,
                                    int64_t ld_out, void* stream) {
  clear_error();
  return vel_at_adjoint(targets, src, lam, ld_lam, dpos, dstr, ld_out, nullptr, 0, stream,
                        "vpm_induced_velocity_at_adjoint");
}

size_t vpm_induced_velocity_at_adjoint_workspace_bytes(int64_t m, int64_t n) {
  return row_workspace_bytes(n, m, OpVelAtAdjoint::kOut);
}

int vpm_induced_velocity_at_adjoint_ws(const vpm_points_t* targets, const vpm_particles_t* src,
                                       const double* lam, int64_t ld_lam, double* dpos,
                                       double* dstr, int64_t ld_out, void* workspace,
                                       size_t ws_bytes, void* stream) {
  clear_error();
  return vel_at_adjoint(targets, src, lam, ld_lam, dpos, dstr, ld_out, workspace, ws_bytes, stream,
                        "vpm_induced_velocity_at_adjoint_ws");
}

}  // extern "C"
