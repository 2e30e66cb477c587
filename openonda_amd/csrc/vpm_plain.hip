// FP64 drop-in kernels: one operator per function of the reference physics
// module, over the row driver (vpm_rows.h).
//
// Reference: OpenONDA/solvers/VPM/ParticlesPhysicsCuda.py (variant CUDA) and
// OpenONDA/solvers/VPM/ParticlesPhysics.py (variant CPU).  The same sums and
// masks in FP64, with the reference's powers and divisions written in one
// inverse root per pair: with s = sigma_ij, D = r^2 + s^2, t = D^-1/2 and
// w = s^2 t^2 (= 1/A of the reference's A = r^2/s^2 + 1),
//   (rho^2 + 2.5) / (A^5/2 s^3)     = t^3 (1 + 1.5 w)
//   3 (rho^2 + 3.5) / (A^7/2 s^5)   = t^5 (3 + 7.5 w)
//   1 / (A^9/2 s^2)                 = s t^3 w^3
//   1 / (A^7/2 s^3)                 = t^3 w^2
//   (r^2 + 3.2 s^2) / D^3/2         = t (1 + 2.2 w),
// so no division and no pow is left (a pair took 200-350 FP64 instructions
// with them and takes 25-45 now).  All factors stay finite wherever the
// reference's powers of s and A do, up to a factor of ten in the lengths.
// Bound: FP64 issue.  One MI355X, before and after (before: one target per
// lane of 256-lane workgroups, so 63 workgroups at N = 16,007, pow and IEEE
// division per pair): driver step with LES and RK2 at N = 16,007 44.3 -> 1.08
// ms, the three scalar sums at N = 20,011 36.6 -> 0.61 ms, velocity and
// vorticity of 16,007 particles at 30,011 points 18.0 -> 0.84 ms, velocity
// and stretching of 1,000 host particles 1.40 -> 0.15 ms with the copies.
// Each operator keeps the reference's per-pair differences and cross products,
// so the rounding of a pair is a few ulp of that pair's own terms.

#include "vpm_rows.h"

namespace vpm {

namespace {

// ---------------------------------------------------------------------------
// Pair operators.  Each has Acc (per-target state), pair() and a result.
// kTargetData: the targets are particles (strength, radius); kRadius, kNu:
// the source data read; kSkipSelf: the reference sums j != i.
// ---------------------------------------------------------------------------

// t^3 (1 + 1.5 w), the velocity and stretching kernel.
struct VelKernel {
  double s2, t, t2, t3, w;
  __device__ __forceinline__ VelKernel(double r2, double s) {
    s2 = s * s;
    t = rsq64(r2 + s2);
    t2 = t * t;
    t3 = t2 * t;
    w = s2 * t2;
  }
  __device__ __forceinline__ double q() const { return t3 * fma(1.5, w, 1.0); }
};

// ParticlesPhysicsCuda.py:65-97 / ParticlesPhysics.py:46-74.
struct OpVelAt {
  static constexpr bool kTargetData = false, kRadius = true, kNu = false, kSkipSelf = false;
  static constexpr int kOut = 3;
  static constexpr bool kSum = false, kSelfTerm = false;
  struct Acc { double ux = 0, uy = 0, uz = 0; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
    if (r2 > kEpsPair) {
      const double q = VelKernel(r2, s.s).q();
      a.ux = fma(q, rz * s.ay - ry * s.az, a.ux);
      a.uy = fma(q, rx * s.az - rz * s.ax, a.uy);
      a.uz = fma(q, ry * s.ax - rx * s.ay, a.uz);
    }
  }
  static __device__ inline void result(const Acc& a, const RowTarget&, double* v) {
    v[0] = a.ux * kOneOverFourPi;
    v[1] = a.uy * kOneOverFourPi;
    v[2] = a.uz * kOneOverFourPi;
  }
};

// CUDA: ParticlesPhysicsCuda.py:159-191 (sigma_ij).  CPU: ParticlesPhysics.py:109-143
// (sigma_i).
template <bool CPUV>
struct OpVelSelf {
  static constexpr bool kTargetData = true, kRadius = !CPUV, kNu = false, kSkipSelf = true;
  static constexpr int kOut = 3;
  static constexpr bool kSum = false, kSelfTerm = false;
  struct Acc { double ux = 0, uy = 0, uz = 0; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
    const double q = VelKernel(r2, CPUV ? t.s : fma(0.5, s.s, t.hs)).q();
    a.ux = fma(q, rz * s.ay - ry * s.az, a.ux);
    a.uy = fma(q, rx * s.az - rz * s.ax, a.uy);
    a.uz = fma(q, ry * s.ax - rx * s.ay, a.uz);
  }
  static __device__ inline void result(const Acc& a, const RowTarget&, double* v) {
    v[0] = kOneOverFourPi * a.ux;
    v[1] = kOneOverFourPi * a.uy;
    v[2] = kOneOverFourPi * a.uz;
  }
};

// CUDA: simplified zeta form, ParticlesPhysicsCuda.py:319-346.
// CPU : full curl form, ParticlesPhysics.py:236-262.
template <bool CPUV>
struct OpVortAt {
  static constexpr bool kTargetData = false, kRadius = true, kNu = false, kSkipSelf = false;
  static constexpr int kOut = 3;
  static constexpr bool kSum = false, kSelfTerm = false;
  struct Acc { double wx = 0, wy = 0, wz = 0; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
    if (r2 > kEpsPair) {
      if constexpr (!CPUV) {  // 7.5 applied in result()
        const double s2 = s.s * s.s;
        const double tt = rsq64_inf(r2 + s2);
        const double t2 = tt * tt, w = s2 * t2;
        const double xi = (t2 * tt) * (w * w);
        a.wx = fma(xi, s.ax, a.wx);
        a.wy = fma(xi, s.ay, a.wy);
        a.wz = fma(xi, s.az, a.wz);
      } else {
        const VelKernel k(r2, s.s);
        const double xi = 7.5 * (k.t3 * (k.w * k.w));
        const double q = k.q();
        const double term1 = xi - q;
        const double term2 = (3.0 * q - xi) * (rx * s.ax + ry * s.ay + rz * s.az) / r2;
        a.wx += term1 * s.ax + term2 * rx;
        a.wy += term1 * s.ay + term2 * ry;
        a.wz += term1 * s.az + term2 * rz;
      }
    }
  }
  static __device__ inline void result(const Acc& a, const RowTarget&, double* v) {
    const double k = CPUV ? kOneOverFourPi : 7.5 * kOneOverFourPi;
    v[0] = a.wx * k;
    v[1] = a.wy * k;
    v[2] = a.wz * k;
  }
};

// ParticlesPhysicsCuda.py:396-445 / ParticlesPhysics.py:291-312.  The sum of
// f1 a_i x a_j is a_i x sum f1 (a_j - a_i): the differences are exact or
// nearly so along tubes and sheets, where a_i x sum f1 a_j would cancel.
struct OpStretch {
  static constexpr bool kTargetData = true, kRadius = true, kNu = false, kSkipSelf = true;
  static constexpr int kOut = 3;
  static constexpr bool kSum = false, kSelfTerm = false;
  struct Acc { double sx = 0, sy = 0, sz = 0, gx = 0, gy = 0, gz = 0; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
    const VelKernel k(r2, fma(0.5, s.s, t.hs));
    const double f1 = k.q();
    a.gx = fma(f1, s.ax - t.ax, a.gx);
    a.gy = fma(f1, s.ay - t.ay, a.gy);
    a.gz = fma(f1, s.az - t.az, a.gz);
    const double cx = ry * s.az - rz * s.ay;
    const double cy = rz * s.ax - rx * s.az;
    const double cz = rx * s.ay - ry * s.ax;
    const double p3 = fma(t.ax, cx, fma(t.ay, cy, t.az * cz));
    const double f2 = (k.t3 * k.t2) * fma(7.5, k.w, 3.0) * p3;
    a.sx = fma(f2, rx, a.sx);
    a.sy = fma(f2, ry, a.sy);
    a.sz = fma(f2, rz, a.sz);
  }
  static __device__ inline void result(const Acc& a, const RowTarget& t, double* v) {
    v[0] = ((t.ay * a.gz - t.az * a.gy) + a.sx) * kOneOverFourPi;
    v[1] = ((t.az * a.gx - t.ax * a.gz) + a.sy) * kOneOverFourPi;
    v[2] = ((t.ax * a.gy - t.ay * a.gx) + a.sz) * kOneOverFourPi;
  }
};

// CUDA: ParticlesPhysicsCuda.py:500-530 (nu_i).  CPU: ParticlesPhysics.py:353-382
// (nu_ij, A + 1e-8, 1/(4pi) once at the end).
template <bool CPUV>
struct OpPse {
  static constexpr bool kTargetData = true, kRadius = true, kNu = true, kSkipSelf = true;
  static constexpr int kOut = 3;
  static constexpr bool kSum = false, kSelfTerm = false;
  struct Acc { double dx = 0, dy = 0, dz = 0; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
    const double sg = fma(0.5, s.s, t.hs);
    const double s2 = sg * sg;
    const double tt = rsq64_inf(CPUV ? fma(s2, 1.0 + kEpsPair, r2) : r2 + s2);
    const double t2 = tt * tt, w = s2 * t2;
    double f3 = (sg * (t2 * tt)) * (w * w * w);
    if constexpr (CPUV) f3 *= t.nu + s.nu;
    a.dx = fma(f3, s.ax - t.ax, a.dx);
    a.dy = fma(f3, s.ay - t.ay, a.dy);
    a.dz = fma(f3, s.az - t.az, a.dz);
  }
  static __device__ inline void result(const Acc& a, const RowTarget& t, double* v) {
    const double k = 105.0 * kOneOverFourPi * (CPUV ? 0.5 : t.nu);
    v[0] = a.dx * k;
    v[1] = a.dy * k;
    v[2] = a.dz * k;
  }
};

// Kinetic energy pair term: ParticlesPhysicsCuda.py:585-631 (CUDA) and
// ParticlesPhysics.py:404-427 (CPU, A + 1e-8).  Scale 1/(16 pi) on the total.
// (2 rho A^-1/2 p1 + rho^3 A^-3/2 (p2 p3 - p1)) / |r| without the division by
// |r|: t (2 - r^2 t^2) p1 + t^3 (r.a_i)(r.a_j).  The reference's unit vector
// r/|r| is NaN for two particles at one point, and so is its energy: kept.
template <bool CPUV>
struct OpEnergy {
  static constexpr bool kTargetData = true, kRadius = true, kNu = false, kDiagonal = false;
  struct Acc { double e = 0; bool nan = false; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
    const double sg = fma(0.5, s.s, t.hs);
    const double tt = rsq64(fma(sg * sg, CPUV ? 1.0 + kEpsPair : 1.0, r2));
    const double t2 = tt * tt;
    const double p1 = fma(t.ax, s.ax, fma(t.ay, s.ay, t.az * s.az));
    const double ri = fma(rx, t.ax, fma(ry, t.ay, rz * t.az));
    const double rj = fma(rx, s.ax, fma(ry, s.ay, rz * s.az));
    a.e = fma(tt, fma(fma(-r2, t2, 2.0), p1, t2 * (ri * rj)), a.e);
    a.nan |= r2 == 0.0;
  }
  static __device__ inline double value(const Acc& a) { return a.nan ? NAN : a.e; }
};

// Helicity pair term: ParticlesPhysicsCuda.py:707-739 (CUDA) and
// ParticlesPhysics.py:448-466 (CPU): one sum, two scales.
struct OpHelicity {
  static constexpr bool kTargetData = true, kRadius = true, kNu = false, kDiagonal = false;
  struct Acc { double h = 0; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
    const double q = VelKernel(r2, fma(0.5, s.s, t.hs)).q();
    const double p1x = t.ay * s.az - t.az * s.ay;
    const double p1y = t.az * s.ax - t.ax * s.az;
    const double p1z = t.ax * s.ay - t.ay * s.ax;
    a.h = fma(fma(rx, p1x, fma(ry, p1y, rz * p1z)), q, a.h);
  }
  static __device__ inline double value(const Acc& a) { return a.h; }
};

// Enstrophy pair term (i = j included): ParticlesPhysicsCuda.py:886-909 and
// ParticlesPhysics.py:533-548.
struct OpEnstrophy {
  static constexpr bool kTargetData = true, kRadius = true, kNu = false, kDiagonal = true;
  struct Acc { double e = 0; };
  static __device__ __forceinline__ void pair(Acc& a, const RowTarget& t, const RowSource& s) {
    const double rx = t.x - s.x, ry = t.y - s.y, rz = t.z - s.z;
    const double r2 = fma(rx, rx, fma(ry, ry, rz * rz));
    const double sg = fma(0.5, s.s, t.hs);
    const double s2 = sg * sg;
    const double tt = rsq64(r2 + s2);
    const double w = s2 * (tt * tt);
    const double p1 = fma(t.ax, s.ax, fma(t.ay, s.ay, t.az * s.az));
    a.e = fma(tt * fma(2.2, w, 1.0), p1, a.e);
  }
  static __device__ inline double value(const Acc& a) { return a.e; }
};

RowArgs args_from(const vpm_particles_t* p) {
  RowArgs a{};
  a.m = a.n = p->n;
  a.tpos = a.pos = p->pos;
  a.tq = a.q = p->str;
  a.tld = a.ld = a.tqld = a.qld = p->ld;
  a.ts = a.s = p->sigma;
  a.tnu = a.nu = p->nu;
  return a;
}

RowArgs args_at(const vpm_points_t* t, const vpm_particles_t* p) {
  RowArgs a = args_from(p);
  a.m = t->m;
  a.tpos = t->pos;
  a.tld = t->ld;
  a.tq = a.ts = a.tnu = nullptr;
  return a;
}

template <class OpCuda, class OpCpu>
int reduce_pair(const vpm_particles_t* p, int variant, double scale_cuda, double scale_cpu,
                double* result, void* ws, size_t ws_bytes, void* stream, const char* who) {
  int rc = check_particles(p, false, who);
  if (rc) return rc;
  if (!result) return fail(VPM_ERR_ARG, "result pointer is null");
  if (variant != VPM_VARIANT_CUDA && variant != VPM_VARIANT_CPU)
    return fail(VPM_ERR_ARG, "unknown variant");
  const size_t need = vpm_reduction_workspace_bytes(p->n);
  if (ws_bytes < need || (need && !ws)) return fail(VPM_ERR_WORKSPACE, "reduction workspace too small");
  hipStream_t st = as_stream(stream);
  double* sums = static_cast<double*>(ws);
  int64_t blocks = 0;
  if (variant == VPM_VARIANT_CUDA)
    rc = row_scalar_launch<OpCuda>(args_from(p), sums, &blocks, st, who);
  else
    rc = row_scalar_launch<OpCpu>(args_from(p), sums, &blocks, st, who);
  if (rc) return rc;
  hipLaunchKernelGGL(final_sum_kernel, dim3(1), dim3(1024), 0, st, sums, blocks,
                     variant == VPM_VARIANT_CUDA ? scale_cuda : scale_cpu, result);
  VPM_LAUNCH_CHECK("final_sum_kernel");
  return VPM_OK;
}

// The sums behind the vector entry points, with or without a workspace.
int vel_at(const vpm_points_t* t, const vpm_particles_t* src, double* out, int64_t ld_out,
           void* ws, size_t ws_bytes, void* stream, const char* who) {
  int rc = check_points(t, who);
  if (rc) return rc;
  if ((rc = check_particles(src, false, who))) return rc;
  if ((rc = check_out(out, ld_out, t->m, who))) return rc;
  RowArgs a = args_at(t, src);
  a.out[0] = out;
  a.ld_out = ld_out;
  return row_launch<OpVelAt>(a, ws, ws_bytes, as_stream(stream), "vel_at");
}

int vort_at(const vpm_points_t* t, const vpm_particles_t* src, int variant, double* out,
            int64_t ld_out, void* ws, size_t ws_bytes, void* stream, const char* who) {
  int rc = check_points(t, who);
  if (rc) return rc;
  if ((rc = check_particles(src, false, who))) return rc;
  if ((rc = check_out(out, ld_out, t->m, who))) return rc;
  RowArgs a = args_at(t, src);
  a.out[0] = out;
  a.ld_out = ld_out;
  if (variant == VPM_VARIANT_CUDA)
    return row_launch<OpVortAt<false>>(a, ws, ws_bytes, as_stream(stream), "vort_at");
  if (variant == VPM_VARIANT_CPU)
    return row_launch<OpVortAt<true>>(a, ws, ws_bytes, as_stream(stream), "vort_at_cpu");
  return fail(VPM_ERR_ARG, "unknown variant");
}

int self_sum(const vpm_particles_t* p, int what, int variant, double* out, int64_t ld_out,
             void* ws, size_t ws_bytes, void* stream, const char* who) {
  int rc = check_particles(p, what == VPM_SUM_PSE, who);
  if (rc) return rc;
  if ((rc = check_out(out, ld_out, p->n, who))) return rc;
  if (variant != VPM_VARIANT_CUDA && variant != VPM_VARIANT_CPU)
    return fail(VPM_ERR_ARG, "unknown variant");
  RowArgs a = args_from(p);
  a.out[0] = out;
  a.ld_out = ld_out;
  hipStream_t st = as_stream(stream);
  const bool cpu = variant == VPM_VARIANT_CPU;
  switch (what) {
    case VPM_SUM_VELOCITY:
      return cpu ? row_launch<OpVelSelf<true>>(a, ws, ws_bytes, st, "vel_self_cpu")
                 : row_launch<OpVelSelf<false>>(a, ws, ws_bytes, st, "vel_self");
    case VPM_SUM_STRETCHING:
      return row_launch<OpStretch>(a, ws, ws_bytes, st, "stretch");
    default:
      return cpu ? row_launch<OpPse<true>>(a, ws, ws_bytes, st, "pse_cpu")
                 : row_launch<OpPse<false>>(a, ws, ws_bytes, st, "pse");
  }
}

}  // namespace

}  // namespace vpm

using namespace vpm;

extern "C" {

size_t vpm_reduction_workspace_bytes(int64_t n) {
  if (n <= 0) return sizeof(double);
  int splits = 1;
  return static_cast<size_t>(row_scalar_blocks(n, &splits)) * sizeof(double);
}

size_t vpm_pair_sum_workspace_bytes(int64_t m, int64_t n) { return row_workspace_bytes(m, n, 3); }

int vpm_pair_sum(const vpm_points_t* targets, const vpm_particles_t* p, int what, int variant,
                 double* out, int64_t ld_out, void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  switch (what) {
    case VPM_SUM_VELOCITY:
      if (targets)
        return vel_at(targets, p, out, ld_out, workspace, ws_bytes, stream, "vpm_pair_sum");
      break;
    case VPM_SUM_VORTICITY:
      return vort_at(targets, p, variant, out, ld_out, workspace, ws_bytes, stream, "vpm_pair_sum");
    case VPM_SUM_STRETCHING:
    case VPM_SUM_PSE:
      if (targets) return fail(VPM_ERR_ARG, "vpm_pair_sum: a self evaluation takes no targets");
      break;
    default:
      return fail(VPM_ERR_ARG, "vpm_pair_sum: unknown sum");
  }
  return self_sum(p, what, variant, out, ld_out, workspace, ws_bytes, stream, "vpm_pair_sum");
}

int vpm_get_induced_velocity_at(const vpm_points_t* targets, const vpm_particles_t* src,
                                double* out, int64_t ld_out, void* stream) {
  clear_error();
  return vel_at(targets, src, out, ld_out, nullptr, 0, stream, "vpm_get_induced_velocity_at");
}

int vpm_get_selfinduced_velocity(const vpm_particles_t* p, int variant, double* out,
                                 int64_t ld_out, void* stream) {
  clear_error();
  return self_sum(p, VPM_SUM_VELOCITY, variant, out, ld_out, nullptr, 0, stream,
                  "vpm_get_selfinduced_velocity");
}

int vpm_get_vorticity_field_at(const vpm_points_t* targets, const vpm_particles_t* src,
                               int variant, double* out, int64_t ld_out, void* stream) {
  clear_error();
  return vort_at(targets, src, variant, out, ld_out, nullptr, 0, stream,
                 "vpm_get_vorticity_field_at");
}

int vpm_get_strength_gradients(const vpm_particles_t* p, double* out, int64_t ld_out,
                               void* stream) {
  clear_error();
  return self_sum(p, VPM_SUM_STRETCHING, VPM_VARIANT_CUDA, out, ld_out, nullptr, 0, stream,
                  "vpm_get_strength_gradients");
}

int vpm_get_strength_gradients_pse(const vpm_particles_t* p, int variant, double* out,
                                   int64_t ld_out, void* stream) {
  clear_error();
  return self_sum(p, VPM_SUM_PSE, variant, out, ld_out, nullptr, 0, stream,
                  "vpm_get_strength_gradients_pse");
}

int vpm_get_total_kinetic_energy(const vpm_particles_t* p, int variant, double* result,
                                 void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  const double k = 1.0 / (16.0 * kPi);
  return reduce_pair<OpEnergy<false>, OpEnergy<true>>(p, variant, k, k, result, workspace,
                                                      ws_bytes, stream, "vpm_get_total_kinetic_energy");
}

int vpm_get_total_helicity(const vpm_particles_t* p, int variant, double* result,
                           void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  return reduce_pair<OpHelicity, OpHelicity>(
      p, variant, kOneOverFourPi * kOneOverFourPi, kOneOverFourPi, result, workspace, ws_bytes,
      stream, "vpm_get_total_helicity");
}

int vpm_get_total_enstrophy(const vpm_particles_t* p, int variant, double* result,
                            void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  const double k8 = 1.0 / (8.0 * kPi);
  return reduce_pair<OpEnstrophy, OpEnstrophy>(p, variant, k8 * kOneOverFourPi, k8, result,
                                               workspace, ws_bytes, stream,
                                               "vpm_get_total_enstrophy");
}

}  // extern "C"
