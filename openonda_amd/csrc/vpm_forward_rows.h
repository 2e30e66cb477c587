// The FP64 row pass behind vpm_forward (vpm_forward_rows.hip).
#pragma once

#include "vpm_common.h"

namespace vpm {

// Sets up to this size run the FP64 rows also in the FP32-compensated
// precision: the FP32 kernels sum pairs two to three times as fast, but their
// sort, records and few target blocks cost 45-100 us first.  Velocity +
// stretching, uniform radius, rows / FP32 kernels: cloud of 2,048 21 / 252 us,
// 4,096 38 / 102, 8,192 102 / 118, 12,288 200 / 193; ring of 4,096 38 / 124,
// 12,288 197 / 250; with PSE 8,192 116 / 148 (ring), vorticity and enstrophy
// 78 / 83.
constexpr int64_t kForwardRowsMax = 8191;

// The FP64 pass always; the FP32-compensated pass for small sets with no
// tile shape and no FP32 sum of G asked for.
inline bool forward_rows_wanted(int64_t n, const vpm_forward_opts_t* o) {
  if (o->precision == VPM_PREC_F64) return true;
  return n <= kForwardRowsMax && o->tile_config < 0 && o->g64_mode != VPM_G64_NEVER;
}

// Bytes of split partials for n particles and the instantiated output set.
size_t forward_rows_split_bytes(int64_t n, unsigned mask);

// The pass; ens_part has room for one double per 64 particles.
int forward_rows(const vpm_particles_t* p, const vpm_forward_opts_t* o, vpm_forward_out_t* out,
                 unsigned mask, double* ens_part, void* split, size_t split_bytes,
                 hipStream_t st);

}  // namespace vpm
