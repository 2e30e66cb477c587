// The FP64 row pass behind vpm_forward (vpm_forward_rows.hip).
#pragma once

#include "vpm_common.h"

namespace vpm {

// Sets up to this size run the FP64 rows also in the FP32-compensated
// precision: the FP32 rows sum pairs up to three times as fast, but first sort
// and write records, and rings leave them few far chunks.  FP64 / FP32 rows,
// uniform radius: velocity, cloud of 4,096 28 / 37 us, 7,000 60 / 55, 9,000
// 85 / 71; velocity + stretching, cloud of 4,096 35 / 54, 8,000 93 / 86, 9,000
// 119 / 107, ring of 8,000 92 / 108, 10,000 143 / 149; with PSE, ring of 8,000
// 109 / 113, 9,000 141 / 141; vorticity + enstrophy + stretching, cloud of
// 8,000 120 / 117, 9,000 156 / 146.
constexpr int64_t kForwardRowsMax = 8191;

// The FP64 pass always; the FP32-compensated pass for small sets with no
// tile shape and no FP32 sum of G asked for.
inline bool forward_rows_wanted(int64_t n, const vpm_forward_opts_t* o) {
  if (o->precision == VPM_PREC_F64) return true;
  return n <= kForwardRowsMax && o->tile_config < 0 && o->g64_mode != VPM_G64_NEVER;
}

// From this size on the FP64 pass reads its particles as packed records, made
// in the call.  The seven arrays of fewer particles (3.6 MB) stay in an XCD's
// 4 MB of L2; of more they do not, and where they lie a multiple of 256 KiB
// apart the seven lines of a source fall into the same cache sets, times the
// eight waves of a workgroup at eight places: velocity of 425,984 particles
// 269 -> 152 ms (tiled FP64 pass 175), of 786,432 1012 -> 517 (592), velocity +
// stretching of 2^19 480 -> 327 (373).  At other strides both forms take the
// same time (400,011 particles 137.4 and 137.1 ms, 100,003 8.5 and 8.6), below
// 65,536 the extra kernel shows (4,096: 50 -> 57 us).
constexpr int64_t kRowRecordsMin = 65536;

// Bytes of split partials for n particles and the instantiated output set.
size_t forward_rows_split_bytes(int64_t n, unsigned mask);

// The pass; ens_part has room for one double per 64 particles.  rec: the
// particles as records in the caller's order, or null (p's arrays are read).
int forward_rows(const vpm_particles_t* p, const Src8* rec, const vpm_forward_opts_t* o,
                 vpm_forward_out_t* out, unsigned mask, double* ens_part, void* split, size_t split_bytes,
                 hipStream_t st);

}  // namespace vpm
