// The fused forward pass in FP64 over the rows of vpm_rows.h: any subset of
// the GPU plugin's outputs from one inverse root per pair, in the caller's
// order (no sort; packed records from kRowRecordsMin particles on).
//
// It is the FP64 pass at every size, and the FP32-compensated pass's stand-in
// for small sets (forward_rows_wanted), where the sort, the records and the
// few target blocks of the FP32 kernels cost more than FP64 arithmetic does.
// Reference arithmetic: ParticlesPhysicsCuda.py:159-191 (velocity), :396-440
// (stretching), :500-525 (PSE), :319-346 (vorticity), :886-909 + :777
// (enstrophy).  Bound: FP64 issue, 37 instructions per pair for velocity +
// stretching with a uniform radius, 41 with sigma_ij.  Velocity + stretching
// of a cloud of 50,021: 4.0 ms with sorted records staged in LDS (80 bytes
// per pair and wave through the LDS return path, which bound it), 3.12 ms
// here (2.98 with kFold); a ring of 4,096 in the FP32-compensated precision
// 131 -> 39 us.

#include "vpm_forward_rows.h"

#include "vpm_rows.h"

namespace vpm {

namespace {

// Powers of one inverse root: D = r^2 + s^2, t = D^-1/2, w = s^2 t^2 (see
// vpm_plain.hip for the factors).
template <unsigned OUT, bool UNIF>
struct OpForward {
  static constexpr bool vel = OUT & VPM_OUT_VEL, str = OUT & VPM_OUT_STRETCH,
                        pse = OUT & VPM_OUT_PSE, vort = OUT & VPM_OUT_VORT,
                        ens = OUT & VPM_OUT_ENSTROPHY;
  static constexpr bool kTargetData = true, kRadius = !UNIF, kNu = pse, kSkipSelf = true;
  static constexpr bool kSum = ens, kSelfTerm = ens;
  static constexpr int kOut = 3 * (vel + str + pse + vort);
  // The set of a solver step with the plain kernels' arithmetic takes the
  // stretching's sum as they do: a_i x sum g (a_j - a_i) (vpm_plain.hip).
  static constexpr bool kDelta = OUT == (VPM_OUT_STRETCH | VPM_OUT_VORT | VPM_OUT_ENSTROPHY);
  // With one radius s the factors' powers of it leave the pair: t^3 (1 + 1.5 w)
  // = t^3 + (1.5 s^2) t^5, and s^2 of the vorticity's t^3 w^2 = s^2 t^5 w and
  // s^3 of PSE's s t^3 w^3 = s^3 t^5 w^2 are applied in result().  Only where
  // the stretching forms t^5 anyway: alone, the others stay finite for radii
  // whose fifth power does not.  Velocity + stretching, 50,021 particles: 3.11
  // -> 2.98 ms for two instructions of 39; a ring of 4,096 39.9 -> 39.4 us.
  static constexpr bool kFold = UNIF && str;
  struct Acc {
    double u[3] = {0, 0, 0}, g[3] = {0, 0, 0}, s[3] = {0, 0, 0}, p[3] = {0, 0, 0},
           w[3] = {0, 0, 0}, e[3] = {0, 0, 0};
  };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double sg = UNIF ? t.s : fma(0.5, s.s, t.hs);
    const double s2 = sg * sg;
    double r2 = 0.0, D;
    if constexpr (vort) {
      r2 = fma(rx, rx, fma(ry, ry, rz * rz));
      D = r2 + s2;
    } else {
      D = fma(rx, rx, fma(ry, ry, fma(rz, rz, s2)));
    }
    // PSE and the vorticity have the reference's weight 0 at infinite distance;
    // the others are inf/inf there
    double t1, t2, t3, t5, w;
    if constexpr (vel || str || pse || ens || UNIF) {
      t1 = (pse || (vort && UNIF)) ? rsq64_inf(D) : rsq64(D);
      t2 = t1 * t1;
      t3 = t2 * t1;
      t5 = t3 * t2;
      w = s2 * t2;
    }
    if constexpr (vel || str) {
      const double g = kFold ? fma(1.5 * s2, t5, t3) : t3 * fma(1.5, w, 1.0);
      const double cx = ry * s.az - rz * s.ay;
      const double cy = rz * s.ax - rx * s.az;
      const double cz = rx * s.ay - ry * s.ax;
      if constexpr (vel) {
        a.u[0] = fma(g, cx, a.u[0]);
        a.u[1] = fma(g, cy, a.u[1]);
        a.u[2] = fma(g, cz, a.u[2]);
      }
      if constexpr (str) {
        a.g[0] = fma(g, kDelta ? s.ax - t.ax : s.ax, a.g[0]);
        a.g[1] = fma(g, kDelta ? s.ay - t.ay : s.ay, a.g[1]);
        a.g[2] = fma(g, kDelta ? s.az - t.az : s.az, a.g[2]);
        const double e = fma(t.ax, cx, fma(t.ay, cy, t.az * cz));
        const double f = t5 * (kFold ? fma(7.5 * s2, t2, 3.0) : fma(7.5, w, 3.0)) * e;
        a.s[0] = fma(f, rx, a.s[0]);
        a.s[1] = fma(f, ry, a.s[1]);
        a.s[2] = fma(f, rz, a.s[2]);
      }
    }
    if constexpr (pse) {
      const double f = kFold ? (t5 * w) * w : (sg * t3) * (w * w * w);
      a.p[0] = fma(f, s.ax - t.ax, a.p[0]);
      a.p[1] = fma(f, s.ay - t.ay, a.p[1]);
      a.p[2] = fma(f, s.az - t.az, a.p[2]);
    }
    if constexpr (vort) {  // sigma_j, not sigma_ij (ParticlesPhysicsCuda.py:323,334-337)
      double x;
      if constexpr (UNIF) {
        x = kFold ? t5 * w : t3 * (w * w);
      } else {
        const double j2 = s.s * s.s;
        const double q1 = rsq64_inf(r2 + j2);
        const double q2 = q1 * q1, wj = j2 * q2;
        x = (q2 * q1) * (wj * wj);
      }
      x = r2 > kEpsPair ? x : 0.0;
      a.w[0] = fma(x, s.ax, a.w[0]);
      a.w[1] = fma(x, s.ay, a.w[1]);
      a.w[2] = fma(x, s.az, a.w[2]);
    }
    if constexpr (ens) {
      const double x = UNIF ? fma(2.2 * s2, t3, t1) : t1 * fma(2.2, w, 1.0);
      a.e[0] = fma(x, s.ax, a.e[0]);
      a.e[1] = fma(x, s.ay, a.e[1]);
      a.e[2] = fma(x, s.az, a.e[2]);
    }
  }
  // the pair i = j, which only the enstrophy sums: r = 0, t = 1/s, w = 1
  static __device__ __forceinline__ void self(Acc& a, const RowTarget& t) {
    const double x = 3.2 / t.s;
    a.e[0] = fma(x, t.ax, a.e[0]);
    a.e[1] = fma(x, t.ay, a.e[1]);
    a.e[2] = fma(x, t.az, a.e[2]);
  }
  static __device__ inline void result(const Acc& a, const RowTarget& t, double* v) {
    constexpr double C = kOneOverFourPi;
    int q = 0;
    if constexpr (vel)
      for (int c = 0; c < 3; ++c) v[q++] = -C * a.u[c];
    if constexpr (str) {
      v[q++] = C * ((t.ay * a.g[2] - t.az * a.g[1]) + a.s[0]);
      v[q++] = C * ((t.az * a.g[0] - t.ax * a.g[2]) + a.s[1]);
      v[q++] = C * ((t.ax * a.g[1] - t.ay * a.g[0]) + a.s[2]);
    }
    if constexpr (pse)
      for (int c = 0; c < 3; ++c)
        v[q++] = 105.0 * t.nu * C * (kFold ? (t.s * t.s * t.s) * a.p[c] : a.p[c]);
    if constexpr (vort)
      for (int c = 0; c < 3; ++c) v[q++] = 7.5 * C * (kFold ? (t.s * t.s) * a.w[c] : a.w[c]);
    if constexpr (ens) v[q++] = fma(t.ax, a.e[0], fma(t.ay, a.e[1], t.az * a.e[2]));
  }
};

template <unsigned OUT, bool UNIF>
int launch(const vpm_particles_t* p, const Src8* rec, const vpm_forward_opts_t* o, vpm_forward_out_t* out,
           double* ens_part, void* split, size_t split_bytes, hipStream_t st) {
  using Op = OpForward<OUT, UNIF>;
  RowArgs a{};
  a.m = a.n = p->n;
  a.tpos = a.pos = p->pos;
  a.tq = a.q = p->str;
  a.tld = a.ld = a.tqld = a.qld = p->ld;
  a.ts = a.s = p->sigma;
  a.tnu = a.nu = p->nu;
  a.rec = rec;
  int v = 0;
  const unsigned want = o->outputs;
  if constexpr (Op::vel) a.out[v++] = (want & VPM_OUT_VEL) ? out->vel : nullptr;
  if constexpr (Op::str) a.out[v++] = (want & VPM_OUT_STRETCH) ? out->stretch : nullptr;
  if constexpr (Op::pse) a.out[v++] = (want & VPM_OUT_PSE) ? out->pse : nullptr;
  if constexpr (Op::vort) a.out[v++] = (want & VPM_OUT_VORT) ? out->vort : nullptr;
  a.ld_out = out->ld;
  a.sums = ens_part;
  double* sums = nullptr;
  int64_t nsums = 0;
  const int rc = row_launch<Op, true>(a, split, split_bytes, st, "forward_rows", o->max_splits,
                                      &sums, &nsums);
  if (rc) return rc;
  if (want & VPM_OUT_ENSTROPHY) {
    const double k = (1.0 / (8.0 * kPi)) * kOneOverFourPi;
    hipLaunchKernelGGL(final_sum_kernel, dim3(1), dim3(1024), 0, st, sums, nsums, k,
                       out->enstrophy);
    VPM_LAUNCH_CHECK("final_sum_kernel");
  }
  return VPM_OK;
}

template <unsigned OUT>
int launch_mode(const vpm_particles_t* p, const Src8* rec, const vpm_forward_opts_t* o,
                vpm_forward_out_t* out, double* ens_part, void* split, size_t split_bytes, hipStream_t st) {
  return o->sigma_mode == VPM_SIGMA_UNIFORM
             ? launch<OUT, true>(p, rec, o, out, ens_part, split, split_bytes, st)
             : launch<OUT, false>(p, rec, o, out, ens_part, split, split_bytes, st);
}

int row_outputs(unsigned mask) {
  int c = 0;
  for (unsigned b = 1; b < VPM_OUT_ENSTROPHY; b <<= 1) c += (mask & b) ? 3 : 0;
  return c;
}

}  // namespace

size_t forward_rows_split_bytes(int64_t n, unsigned mask) {
  return row_workspace_bytes(n, n, row_outputs(mask), (mask & VPM_OUT_ENSTROPHY) != 0);
}

int forward_rows(const vpm_particles_t* p, const Src8* rec, const vpm_forward_opts_t* o,
                 vpm_forward_out_t* out, unsigned mask, double* ens_part, void* split, size_t split_bytes,
                 hipStream_t st) {
  switch (mask) {
#define VPM_ROWS(M) \
  case M: return launch_mode<M>(p, rec, o, out, ens_part, split, split_bytes, st);
    VPM_ROWS(1u) VPM_ROWS(2u) VPM_ROWS(3u) VPM_ROWS(4u) VPM_ROWS(7u) VPM_ROWS(8u) VPM_ROWS(16u)
    VPM_ROWS(24u) VPM_ROWS(26u)
    VPM_ROWS(27u)
#undef VPM_ROWS
    default: return launch_mode<31u>(p, rec, o, out, ens_part, split, split_bytes, st);
  }
}

}  // namespace vpm
