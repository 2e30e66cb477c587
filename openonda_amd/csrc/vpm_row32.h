// The FP32-compensated row pass behind vpm_forward (vpm_row32.hip).
#pragma once

#include "vpm_pass.h"

namespace vpm {

// Output sets and radius modes the row pass runs when no tile shape is asked
// for: those without the far-field moment form (it needs velocity, stretching
// and a uniform radius).
inline bool row32_wanted(unsigned mask, bool unif, const vpm_forward_opts_t* o) {
  const bool moment = unif && (mask & VPM_OUT_VEL) && (mask & VPM_OUT_STRETCH);
  return o->precision == VPM_PREC_F32C && o->tile_config < 0 && !moment;
}

// Bytes of the FP32 records, the chunk boxes and the split partials.
size_t row32_record_bytes(int64_t n);
size_t row32_box_bytes(int64_t n);
size_t row32_split_bytes(int64_t n, unsigned mask);

// Builds the records from the sorted particles a.src and runs the pass;
// *nblocks: enstrophy partials written to a.ens_part.
int row32_run(const FusedArgs& a, unsigned mask, bool unif, float* rec, double* box,
              hipStream_t st, int* nblocks);

}  // namespace vpm
