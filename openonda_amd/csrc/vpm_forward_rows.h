// The FP64 row pass behind vpm_forward (vpm_forward_rows.hip).
#pragma once

#include "vpm_common.h"

namespace vpm {

// Sets up to this size run the FP64 rows also in the FP32-compensated
// precision: the FP32 rows sum pairs up to three times as fast, but first sort
// and write records, and their near chunks fill with few particles.  FP64 /
// FP32 rows, uniform radius: velocity, ring of 2,000 21 / 46 us, 8,000 69 /
// 80, 10,000 102 / 98; velocity + stretching, cloud of 4,000 35 / 67, 8,000
// 92 / 107, 10,000 144 / 138, ring of 8,000 92 / 132, 10,000 142 / 168;
// vorticity + enstrophy + stretching, cloud of 8,000 120 / 140, 10,000 187 /
// 184, general radii 8,000 150 / 155, 10,000 236 / 212.
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
