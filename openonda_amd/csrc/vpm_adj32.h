// The FP32-compensated adjoint over rows (vpm_adj32.hip).
#pragma once

#include "vpm_common.h"

namespace vpm {

struct Adj32Args {
  vpm_particles_t p;
  const double* lam;    // cotangents [3][ldc], null: zero
  const double* mu;
  const double* xi;
  int64_t ldc;
  const int* perm;      // sorted k -> caller index, or null
  double* dpos;
  double* dstr;
  int64_t ld;
  float* rec;           // adj32_record_bytes
  double* box;          // adj32_box_bytes
  double* part;         // split partials, or null
  size_t part_cap;
  int max_splits;       // 0: automatic
  bool unif;            // one radius
};

size_t adj32_record_bytes(int64_t n);
size_t adj32_box_bytes(int64_t n);
size_t adj32_split_bytes(int64_t n);

// mask: VPM_OUT_VEL | STRETCH | PSE, the cotangents present.
int adj32_run(const Adj32Args& a, unsigned mask, hipStream_t st);

}  // namespace vpm
