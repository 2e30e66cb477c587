// FP32-compensated adjoint over rows of 64 sorted particles (vpm_adjoint.hip
// derives the formulas; the row scheme is that of vpm_row32.hip).
//
// A workgroup owns one row; its eight waves take the partner chunks in turn
// and read the partners' FP32 records, relative to their chunk's centre,
// through scalar loads.  The FP32 sums of a chunk are folded in FP64 into the
// six numbers the particle needs (dL/dx, dL/dalpha), so neither 21 FP64
// totals per lane nor 21 split partials are kept.
//
// With r = x_m - x_j, sc = 1/sigma (lengths are in units of a uniform radius;
// with per-particle radii as they are, sc = 1), per pair
//   near: c = r x a_j, k = lam_j x r - sc Q_j,
//         E = lam_m.c - a_m.k + a_j.(sc P_m), psi = a_m.c
//   far (box gap above 4 radii), with m_j = a_j x x_j, v_j = lam_j x x_j + sc Q_j
//   and p = a_m x x_m relative to the chunk's centre:
//         E = a_j.(lam_m x x_m + sc P_m) + lam_m.m_j + lam_j.p + a_m.v_j,
//         psi = a_j.p + a_m.m_j,
// where sum g k = Lam x x_m - sum g v_j and sum f phi c = x_m x Y + sum f phi m_j
// per chunk: no cross product per pair is left.  81 VALU instructions per far
// pair with all three cotangents, 92 per near one (105 before, all pairs).
// The pair j = m is left out (each of its terms cancels or vanishes).
//
// Bound: FP32 issue.  All three cotangents, against 256-partner tiles in LDS
// with 21 FP64 totals per lane: ring of 131,072 36.2 -> 27.9 ms (rel-L2 of
// dL/dx 5.8e-8 -> 5.4e-8, of dL/dalpha 2.8e-7 -> 1.8e-7), of 2,000 0.110 ->
// 0.063 ms; velocity and stretching only 30.9 -> 22.2 ms; per-particle radii,
// 40,000 particles 3.75 -> 2.9 ms.

#include "vpm_adj32.h"

#include <algorithm>
#include <type_traits>

#include "vpm_rows.h"

namespace vpm {

namespace {

constexpr int kAdjChunk = 64;
// Record: offset 0, a 3, lam 6, mu 9, z = nu xi 12, sigma/2 15, sc Q 16,
// m 19, v 22, a.z 25.
constexpr int kAdjStride = 28;
constexpr int kAdjBox = 8;   // centre, half-extent, largest radius
constexpr int kAdjOut = 6;   // dL/dx, dL/dalpha
constexpr double kAdjGap = 4.0;
// Sources per FP32 run before its sums are folded in FP64: 32 on near chunks,
// whose partial sums' roundings set the error (ring of 131,072: dL/dx 6.9e-8
// with 64, 5.4e-8 with 32), a whole chunk on far ones (5.4e-8 either way; 32
// costs 29.4 ms instead of 27.9).
constexpr int kAdjNearRun = 32, kAdjFarRun = kAdjChunk;
// Waves per SIMD the registers must allow: six with some of the chunk set-up
// in scratch ran 27.8 ms against 29.4 ms for four without.
constexpr int kAdjWaves = 6;

typedef __attribute__((address_space(4))) const float scalar_float_t;

__device__ __forceinline__ double held(double v) {  // rounded here, not fused into its use
  asm volatile("" : "+v"(v));
  return v;
}

__device__ __forceinline__ double adj_scale(const Adj32Args& A) {
  return A.unif ? 1.0 / A.p.sigma[0] : 1.0;
}

// A particle's data in FP64, by sorted index.
struct AdjParticle {
  double x[3], a[3], l[3], m[3], z[3], s;
};

__device__ __forceinline__ AdjParticle adj_particle(const Adj32Args& A, int k) {
  const int64_t i = A.perm ? A.perm[k] : k;
  AdjParticle g;
  const double nu = A.xi ? A.p.nu[i] : 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    g.x[c] = A.p.pos[c * A.p.ld + i];
    g.a[c] = A.p.str[c * A.p.ld + i];
    g.l[c] = A.lam ? A.lam[c * A.ldc + i] : 0.0;
    g.m[c] = A.mu ? A.mu[c * A.ldc + i] : 0.0;
    g.z[c] = A.xi ? nu * A.xi[c * A.ldc + i] : 0.0;
  }
  g.s = A.p.sigma[i];
  return g;
}

__device__ __forceinline__ void cross(const double* a, const double* b, double* o) {
  o[0] = a[1] * b[2] - a[2] * b[1];
  o[1] = a[2] * b[0] - a[0] * b[2];
  o[2] = a[0] * b[1] - a[1] * b[0];
}

// One wave per chunk; lanes past n write zero data far away (every term
// vanishes; PSE's powers of t underflow to 0 at that distance).  The box is
// that of the finite coordinates, as in vpm_row32.hip.
__global__ __launch_bounds__(kAdjChunk) void adj32_records_kernel(Adj32Args A) {
  const int c = blockIdx.x, n = static_cast<int>(A.p.n);
  const int k = c * kAdjChunk + static_cast<int>(threadIdx.x);
  const bool ok = k < n;
  const double scale = adj_scale(A);
  AdjParticle g{};
  if (ok) g = adj_particle(A, k);
  double x[3], cen[3];
  double* box = A.box + static_cast<int64_t>(c) * kAdjBox;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    x[q] = held(g.x[q] * scale);
    const bool in = ok && isfinite(x[q]);
    const double lo = wave_min(in ? x[q] : INFINITY), hi = wave_max(in ? x[q] : -INFINITY);
    cen[q] = lo <= hi ? 0.5 * (lo + hi) : 0.0;
    x[q] -= cen[q];
    if (threadIdx.x == 0) {
      box[q] = cen[q];
      box[3 + q] = lo <= hi ? 0.5 * (hi - lo) : 0.0;
    }
  }
  const double big = wave_max(ok ? g.s * scale : 0.0);
  if (threadIdx.x == 0) {
    box[6] = big;
    box[7] = 0.0;
  }
  double Q[3], m[3], l[3];
  cross(g.a, g.m, Q);
  cross(g.a, x, m);
  cross(g.l, x, l);
  float* r = A.rec + static_cast<int64_t>(k) * kAdjStride;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    r[q] = ok ? static_cast<float>(x[q]) : 1e18f;
    r[3 + q] = static_cast<float>(g.a[q]);
    r[6 + q] = static_cast<float>(g.l[q]);
    r[9 + q] = static_cast<float>(g.m[q]);
    r[12 + q] = static_cast<float>(g.z[q]);
    r[16 + q] = static_cast<float>(scale * Q[q]);
    r[19 + q] = ok ? static_cast<float>(m[q]) : 0.0f;
    r[22 + q] = ok ? static_cast<float>(l[q] + scale * Q[q]) : 0.0f;
  }
  r[15] = ok ? static_cast<float>(0.5 * g.s * scale) : 0.5f;
  r[25] = static_cast<float>(g.a[0] * g.z[0] + g.a[1] * g.z[1] + g.a[2] * g.z[2]);
  r[26] = r[27] = 0.0f;
}

__device__ __forceinline__ void add_cross(double* o, const double* a, const double* b) {
  o[0] = fma(-a[2], b[1], fma(a[1], b[2], o[0]));
  o[1] = fma(-a[0], b[2], fma(a[2], b[0], o[1]));
  o[2] = fma(-a[1], b[0], fma(a[0], b[1], o[2]));
}

struct AdjT32 {
  float x[3], a[3], l[3], m[3], z[3], P[3], hs, az;  // P: sc a x mu; az: a.z
};

// Constants in VGPRs (literal operands halve an instruction's issue rate);
// h75, h2625 carry the factor -2 sc of their term.
struct AdjK {
  float c15, c3, c75, c105, c945, h75, h2625, c45;
};

// FP32 sums of a chunk: G = g a_j, L = g lam_j, A, B, X, Y = f phi a_j,
// D = f psi (mu_m - mu_j), T = 105 p (far form).
struct AdjAcc {
  float G[3], L[3], A[3], B[3], X[3], Y[3], D[3], T;
};

struct AdjW {  // the pair's distance weights
  float d[3], g, f, h, p, q;
};

__device__ __forceinline__ float dot3(const float* a, const float* b, float c) {
  return __builtin_fmaf(a[2], b[2], __builtin_fmaf(a[1], b[1], __builtin_fmaf(a[0], b[0], c)));
}
__device__ __forceinline__ void add3(float* s, float w, const float* v) {
  s[0] = __builtin_fmaf(w, v[0], s[0]);
  s[1] = __builtin_fmaf(w, v[1], s[1]);
  s[2] = __builtin_fmaf(w, v[2], s[2]);
}

template <unsigned OUT, bool UNIF>
__device__ __forceinline__ void adj_weights(AdjW& w_, const AdjT32& t, const float* f,
                                            const AdjK& k, bool self) {
  constexpr bool vs = OUT & (VPM_OUT_VEL | VPM_OUT_STRETCH);
  const float* d = w_.d;
  float s = 1.0f, s2 = 1.0f;
  if constexpr (!UNIF) {
    s = t.hs + f[15];
    s2 = s * s;
  }
  const float D = dot3(d, d, s2);
  float t1 = __builtin_amdgcn_rsqf(D);
  if constexpr (vs)
    if (self) t1 = 0.0f;  // all weights 0, also where a small radius' t7 is infinite
  const float t2 = t1 * t1, t3 = t2 * t1, t5 = t3 * t2;
  const float w = UNIF ? t2 : s2 * t2;
  if constexpr (vs) {
    w_.g = UNIF ? __builtin_fmaf(k.c15, t5, t3) : t3 * __builtin_fmaf(k.c15, w, 1.0f);
    w_.f = t5 * __builtin_fmaf(k.c75, w, k.c3);
  }
  if constexpr ((OUT & VPM_OUT_STRETCH) != 0)
    w_.h = (t5 * t2) * __builtin_fmaf(k.h2625, w, k.h75);
  if constexpr ((OUT & VPM_OUT_PSE) != 0) {
    if constexpr (UNIF) {
      w_.p = (t5 * t2) * t2;
    } else {  // as in vpm_row32.hip: 1 - D t2 takes t2's roundings out of its powers
      const float r = fminf(__builtin_fmaf(-D, t2, 1.0f), 1.0f);
      w_.p = ((s * t3) * (w * w * w)) * __builtin_fmaf(k.c45, r, 1.0f);
    }
    w_.q = w_.p * t2;
  }
}

template <unsigned OUT>
__device__ __forceinline__ void adj_near(AdjAcc& acc, const AdjW& w, const AdjT32& t,
                                         const float* f, const AdjK& k) {
  constexpr bool vel = OUT & VPM_OUT_VEL, str = OUT & VPM_OUT_STRETCH, pse = OUT & VPM_OUT_PSE;
  const float* d = w.d;
  const float *a = f + 3, *l = f + 6, *m = f + 9, *z = f + 12, *Q = f + 16;
  float xc = 0.0f;
  if constexpr (vel || str) {
    const float c[3] = {d[1] * a[2] - d[2] * a[1], d[2] * a[0] - d[0] * a[2],
                        d[0] * a[1] - d[1] * a[0]};
    add3(acc.G, w.g, a);
    float kk[3] = {0.0f, 0.0f, 0.0f}, E = 0.0f;
    if constexpr (vel) {
      kk[0] = l[1] * d[2] - l[2] * d[1];
      kk[1] = l[2] * d[0] - l[0] * d[2];
      kk[2] = l[0] * d[1] - l[1] * d[0];
      add3(acc.L, w.g, l);
      E = dot3(t.l, c, 0.0f);
    }
    if constexpr (str) {
      kk[0] -= Q[0];
      kk[1] -= Q[1];
      kk[2] -= Q[2];
      E = dot3(t.P, a, E);
    }
    add3(acc.A, w.g, kk);
    E -= dot3(t.a, kk, 0.0f);
    xc = w.f * E;
    if constexpr (str) {
      const float dm[3] = {t.m[0] - m[0], t.m[1] - m[1], t.m[2] - m[2]};
      const float phi = dot3(dm, d, 0.0f), psi = dot3(t.a, c, 0.0f);
      const float fphi = w.f * phi;
      add3(acc.B, fphi, c);
      add3(acc.Y, fphi, a);
      add3(acc.D, w.f * psi, dm);
      xc = __builtin_fmaf(w.h * psi, phi, xc);
    }
  }
  if constexpr (pse) {
    const float dz[3] = {z[0] - t.z[0], z[1] - t.z[1], z[2] - t.z[2]};
    const float da[3] = {a[0] - t.a[0], a[1] - t.a[1], a[2] - t.a[2]};
    add3(acc.A, k.c105 * w.p, dz);
    xc = __builtin_fmaf(k.c945 * w.q, dot3(da, dz, 0.0f), xc);
  }
  add3(acc.X, xc, d);
}

// p = a_m x x_m, e = lam_m x x_m + sc P_m, about the chunk's centre.
template <unsigned OUT>
__device__ __forceinline__ void adj_far(AdjAcc& acc, const AdjW& w, const AdjT32& t,
                                        const float* p, const float* e, const float* f,
                                        const AdjK& k) {
  constexpr bool vel = OUT & VPM_OUT_VEL, str = OUT & VPM_OUT_STRETCH, pse = OUT & VPM_OUT_PSE;
  const float* d = w.d;
  const float *a = f + 3, *l = f + 6, *m = f + 9, *z = f + 12, *mo = f + 19, *v = f + 22;
  float xc = 0.0f;
  if constexpr (vel || str) {
    add3(acc.G, w.g, a);
    add3(acc.A, -w.g, v);
    float E = dot3(e, a, 0.0f);
    E = dot3(t.a, v, E);
    if constexpr (vel) {
      add3(acc.L, w.g, l);
      E = dot3(t.l, mo, E);
      E = dot3(p, l, E);
    }
    xc = w.f * E;
    if constexpr (str) {
      const float dm[3] = {t.m[0] - m[0], t.m[1] - m[1], t.m[2] - m[2]};
      const float phi = dot3(dm, d, 0.0f);
      const float psi = dot3(t.a, mo, dot3(p, a, 0.0f));
      const float fphi = w.f * phi;
      add3(acc.B, fphi, mo);
      add3(acc.Y, fphi, a);
      add3(acc.D, w.f * psi, dm);
      xc = __builtin_fmaf(w.h * psi, phi, xc);
    }
  }
  if constexpr (pse) {  // (a_j - a_m).(z_j - z_m) and 105 p (z_j - z_m), expanded
    const float p105 = k.c105 * w.p;
    add3(acc.A, p105, z);
    acc.T += p105;
    float dd = t.az + f[25];
    dd -= dot3(t.a, z, dot3(t.z, a, 0.0f));
    xc = __builtin_fmaf(k.c945 * w.q, dd, xc);
  }
  add3(acc.X, xc, d);
}

// grid (rows, splits)
template <unsigned OUT, bool UNIF>
__global__ __launch_bounds__(kRowBlock, kAdjWaves) void adj32_kernel(Adj32Args A, int splits,
                                                                     int64_t pld) {
  constexpr bool vel = OUT & VPM_OUT_VEL, str = OUT & VPM_OUT_STRETCH, pse = OUT & VPM_OUT_PSE;
  __shared__ double tot[kRowWaves][kAdjOut][kRow];  // per wave: touched once per chunk
  __shared__ double tgt[9][kRow];                   // a, lam, sc mu of the row in FP64
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = blockIdx.x, n = static_cast<int>(A.p.n);
  const int kt = row * kRow + lane;
  const bool valid = kt < n;
  const double scale = adj_scale(A);
  AdjParticle g{};
  g.s = 1.0;
  if (valid) g = adj_particle(A, kt);
  const double X[3] = {held(g.x[0] * scale), held(g.x[1] * scale), held(g.x[2] * scale)};
  AdjT32 t;
  {
    double P[3];
    cross(g.a, g.m, P);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      t.a[q] = static_cast<float>(g.a[q]);
      t.l[q] = static_cast<float>(g.l[q]);
      t.m[q] = static_cast<float>(g.m[q]);
      t.z[q] = static_cast<float>(g.z[q]);
      t.P[q] = static_cast<float>(scale * P[q]);
      if (wave == 0) {
        tgt[q][lane] = g.a[q];
        tgt[3 + q][lane] = g.l[q];
        tgt[6 + q][lane] = scale * g.m[q];
      }
    }
    t.hs = static_cast<float>(0.5 * g.s * scale);
    t.az = static_cast<float>(g.a[0] * g.z[0] + g.a[1] * g.z[1] + g.a[2] * g.z[2]);
  }
  double cen[3], half[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const double lo = wave_min(valid ? X[q] : INFINITY), hi = wave_max(valid ? X[q] : -INFINITY);
    cen[q] = 0.5 * (lo + hi);
    half[q] = 0.5 * (hi - lo);
  }
  const double smax = wave_max(valid ? g.s * scale : 0.0);
#pragma unroll
  for (int q = 0; q < kAdjOut; ++q) tot[wave][q][lane] = 0.0;
  __syncthreads();

  AdjK k{1.5f, 3.0f, 7.5f, 105.0f, 945.0f, static_cast<float>(-15.0 * scale),
         static_cast<float>(-52.5 * scale), 4.5f};
  asm volatile("" : "+v"(k.c15), "+v"(k.c3), "+v"(k.c75), "+v"(k.c105), "+v"(k.c945),
               "+v"(k.h75), "+v"(k.h2625));
  if constexpr (pse && !UNIF) asm volatile("" : "+v"(k.c45));
  AdjAcc acc{};
  const int nchunk = (n + kAdjChunk - 1) / kAdjChunk;
  const int parts = splits * kRowWaves;
  uint64_t near = 0;  // this wave's next 64 chunks near the row
  int seen = 0;
  for (int c = static_cast<int>(blockIdx.y) * kRowWaves + wave; c < nchunk; c += parts, ++seen) {
    if ((seen & 63) == 0) {
      const int64_t cc = c + static_cast<int64_t>(lane) * parts;
      bool nr = false;
      if (cc < nchunk) {
        const double* box = A.box + cc * kAdjBox;
        double gap2 = 0.0;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const double gp = fmax(fabs(box[q] - cen[q]) - half[q] - box[3 + q], 0.0);
          gap2 += gp * gp;
        }
        const double lim = kAdjGap * fmax(smax, box[6]);
        nr = !(gap2 > lim * lim);
      }
      near = __ballot(nr);
    }
    const bool is_near = ((near >> (seen & 63)) & 1u) != 0;
    const scalar_double_t* box =
        (const scalar_double_t*)(A.box + static_cast<int64_t>(c) * kAdjBox);
    double xc[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      xc[q] = X[q] - box[q];
      t.x[q] = static_cast<float>(xc[q]);
    }
    const scalar_float_t* rec =
        (const scalar_float_t*)(A.rec + static_cast<int64_t>(c) * kAdjChunk * kAdjStride);
    auto load = [&](float* b, int q) {
#pragma unroll
      for (int u = 0; u < kAdjStride; ++u) b[u] = rec[q * kAdjStride + u];
    };
    // Two records in registers: the next one's loads issue once the first
    // instructions of the current pair have waited for its own (scalar loads
    // return out of order, so a wait covers every load in flight).  The last
    // reads one record of padding.
    auto stream = [&](auto pair, int q0, int q1, bool own) {
      float bA[kAdjStride], bB[kAdjStride];
      auto one = [&](const float* b, float* nb, int q) {
        AdjW w;
        w.d[0] = t.x[0] - b[0];
        w.d[1] = t.x[1] - b[1];
        w.d[2] = t.x[2] - b[2];
        __builtin_amdgcn_sched_barrier(0);
        load(nb, q + 1);
        __builtin_amdgcn_sched_barrier(0);
        adj_weights<OUT, UNIF>(w, t, b, k, own && q == lane);
        pair(w, b);
      };
      load(bA, q0);
#pragma unroll 1
      for (int q = q0; q < q1; q += 2) {
        one(bA, bB, q);
        one(bB, bA, q + 1);
      }
    };
    // A run's sums in FP64: dA' = A + sc (G x mu + B), dX' = X - G x lam +
    // a x Lam + sc (Y x a + D), and the far form's Lam x x + sc x x Y - z T.
    auto fold = [&](auto far) {
      double dA[3] = {acc.A[0], acc.A[1], acc.A[2]}, dX[3] = {acc.X[0], acc.X[1], acc.X[2]};
      const double G[3] = {acc.G[0], acc.G[1], acc.G[2]};
      const double a[3] = {tgt[0][lane], tgt[1][lane], tgt[2][lane]};
      if constexpr (vel) {
        const double L[3] = {acc.L[0], acc.L[1], acc.L[2]};
        const double l[3] = {tgt[3][lane], tgt[4][lane], tgt[5][lane]};
        if constexpr (far) add_cross(dA, L, xc);
        add_cross(dX, l, G);
        add_cross(dX, a, L);
      }
      if constexpr (str) {
        const double Y[3] = {scale * acc.Y[0], scale * acc.Y[1], scale * acc.Y[2]};
        const double m[3] = {tgt[6][lane], tgt[7][lane], tgt[8][lane]};  // sc mu
        add_cross(dA, G, m);
        if constexpr (far) add_cross(dA, xc, Y);
        add_cross(dX, Y, a);
        for (int q = 0; q < 3; ++q) {
          dA[q] = fma(scale, static_cast<double>(acc.B[q]), dA[q]);
          dX[q] = fma(scale, static_cast<double>(acc.D[q]), dX[q]);
        }
      }
      if constexpr (pse && far) {
        const double T = acc.T;
        for (int q = 0; q < 3; ++q) dA[q] = fma(-static_cast<double>(t.z[q]), T, dA[q]);
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        tot[wave][q][lane] += dX[q];
        tot[wave][3 + q][lane] += dA[q];
      }
      acc = AdjAcc{};
    };
    if (is_near || c == row) {
#pragma unroll 1
      for (int q = 0; q < kAdjChunk; q += kAdjNearRun) {
        stream([&](const AdjW& w, const float* f) { adj_near<OUT>(acc, w, t, f, k); }, q,
               q + kAdjNearRun, c == row);
        fold(std::false_type{});
      }
    } else {
      const float* x = t.x;
      const float p[3] = {t.a[1] * x[2] - t.a[2] * x[1], t.a[2] * x[0] - t.a[0] * x[2],
                          t.a[0] * x[1] - t.a[1] * x[0]};
      float e[3] = {0.0f, 0.0f, 0.0f};
      if constexpr (vel) {
        e[0] = t.l[1] * x[2] - t.l[2] * x[1];
        e[1] = t.l[2] * x[0] - t.l[0] * x[2];
        e[2] = t.l[0] * x[1] - t.l[1] * x[0];
      }
      if constexpr (str) {
        e[0] += t.P[0];
        e[1] += t.P[1];
        e[2] += t.P[2];
      }
#pragma unroll 1
      for (int q = 0; q < kAdjChunk; q += kAdjFarRun) {
        stream([&](const AdjW& w, const float* f) { adj_far<OUT>(acc, w, t, p, e, f, k); }, q,
               q + kAdjFarRun, false);
        fold(std::true_type{});
      }
    }
  }
  __syncthreads();
  if (wave >= kAdjOut) return;  // one wave per component
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) s += tot[w][wave][lane];
  if (A.part) {
    A.part[(static_cast<int64_t>(blockIdx.y) * kAdjOut + wave) * pld + kt] = s;
  } else if (valid) {
    const int64_t o = A.perm ? A.perm[kt] : kt;
    const double s2 = scale * scale;
    if (wave < 3) A.dpos[wave * A.ld + o] = kOneOverFourPi * s2 * scale * s;
    else A.dstr[(wave - 3) * A.ld + o] = kOneOverFourPi * s2 * s;
  }
}

// Adds the splits in order and stores.  grid (particles / 256, 6).
__global__ __launch_bounds__(256) void adj32_reduce_kernel(Adj32Args A, int splits, int64_t pld) {
  const int k = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  const int q = blockIdx.y;
  if (k >= A.p.n) return;
  double s = 0.0;
  for (int i = 0; i < splits; ++i) s += A.part[(static_cast<int64_t>(i) * kAdjOut + q) * pld + k];
  const double scale = adj_scale(A), s2 = scale * scale;
  const int64_t o = A.perm ? A.perm[k] : k;
  if (q < 3) A.dpos[q * A.ld + o] = kOneOverFourPi * s2 * scale * s;
  else A.dstr[(q - 3) * A.ld + o] = kOneOverFourPi * s2 * s;
}

template <unsigned OUT, bool UNIF>
int launch(Adj32Args a, hipStream_t st) {
  const int rows = static_cast<int>(row_count(a.p.n));
  const int chunks = static_cast<int>(ceil_div(a.p.n, kAdjChunk));
  const size_t per = static_cast<size_t>(kAdjOut) * rows * kRow * sizeof(double);
  int k = std::min(row_splits(rows, a.p.n), std::max(1, chunks / kRowWaves));
  if (a.max_splits > 0) k = std::min(k, a.max_splits);
  if (!a.part || a.part_cap / per < 2) k = 1;
  else k = static_cast<int>(std::min<size_t>(k, a.part_cap / per));
  if (k == 1) a.part = nullptr;
  const int64_t pld = static_cast<int64_t>(rows) * kRow;
  hipLaunchKernelGGL(adj32_records_kernel, dim3(chunks), dim3(kAdjChunk), 0, st, a);
  VPM_LAUNCH_CHECK("adj32_records_kernel");
  hipLaunchKernelGGL((adj32_kernel<OUT, UNIF>), dim3(rows, k), dim3(kRowBlock), 0, st, a, k, pld);
  VPM_LAUNCH_CHECK("adj32_kernel");
  if (k > 1) {
    hipLaunchKernelGGL(adj32_reduce_kernel,
                       dim3(static_cast<unsigned>(ceil_div(a.p.n, 256)), kAdjOut), dim3(256), 0, st,
                       a, k, pld);
    VPM_LAUNCH_CHECK("adj32_reduce_kernel");
  }
  return VPM_OK;
}

template <bool UNIF>
int launch_mask(const Adj32Args& a, unsigned mask, hipStream_t st) {
  switch (mask) {
    case 1u: return launch<1u, UNIF>(a, st);
    case 2u: return launch<2u, UNIF>(a, st);
    case 3u: return launch<3u, UNIF>(a, st);
    case 4u: return launch<4u, UNIF>(a, st);
    case 5u: return launch<5u, UNIF>(a, st);
    case 6u: return launch<6u, UNIF>(a, st);
    default: return launch<7u, UNIF>(a, st);
  }
}

}  // namespace

// Records of whole chunks, and one read ahead past the last.
size_t adj32_record_bytes(int64_t n) {
  return (static_cast<size_t>(ceil_div(n > 0 ? n : 1, kAdjChunk)) * kAdjChunk + 1) * kAdjStride *
         sizeof(float);
}

size_t adj32_box_bytes(int64_t n) {
  return static_cast<size_t>(ceil_div(n > 0 ? n : 1, kAdjChunk)) * kAdjBox * sizeof(double);
}

size_t adj32_split_bytes(int64_t n) {
  const int64_t rows = row_count(n);
  const int k = row_splits(rows, n);
  return k > 1 ? static_cast<size_t>(k) * kAdjOut * rows * kRow * sizeof(double) : 0;
}

int adj32_run(const Adj32Args& a, unsigned mask, hipStream_t st) {
  return a.unif ? launch_mask<true>(a, mask, st) : launch_mask<false>(a, mask, st);
}

}  // namespace vpm
