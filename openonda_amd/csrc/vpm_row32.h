// The FP32-compensated row pass behind vpm_forward (vpm_row32.hip).
#pragma once

#include "vpm_pass.h"

namespace vpm {

// The row pass runs every FP32-compensated call that asks for no tile shape
// (vpm_row32.hip has both sides measured), but two output sets that sum in FP64
// on every chunk, where many particles no longer fit the L2: each row reads
// them all again, where the tiled kernels read them once for 256 or 512
// targets.  The stretching alone with a uniform radius, tiled / rows, ms: ring
// of 131,072 15.4 / 14.4, 163,840 21.5 / 23.1, 400,009 135 / 160; cloud of
// 131,072 11.2 / 11.0, 163,840 16.3 / 17.3.  PSE with vorticity or enstrophy and
// per-particle radii: ring of 262,144 121 / 117, 400,009 286 / 298.
constexpr int64_t kRow32StretchMax = 131072, kRow32AllMax = 262144;

inline bool row32_wanted(int64_t n, const vpm_forward_opts_t* o) {
  if (o->precision != VPM_PREC_F32C || o->tile_config >= 0) return false;
  if (o->sigma_mode == VPM_SIGMA_UNIFORM)
    return n <= kRow32StretchMax || o->outputs != VPM_OUT_STRETCH;
  return n <= kRow32AllMax || !(o->outputs & VPM_OUT_PSE) ||
         !(o->outputs & (VPM_OUT_VORT | VPM_OUT_ENSTROPHY));
}

// Bytes of the FP32 records, the chunk boxes and the split partials.
size_t row32_record_bytes(int64_t n);
size_t row32_box_bytes(int64_t n);
size_t row32_split_bytes(int64_t n, unsigned mask, bool unif);

// Builds the records from the sorted particles a.src and runs the pass;
// *nblocks: enstrophy partials written to a.ens_part.
int row32_run(const FusedArgs& a, unsigned mask, bool unif, float* rec, double* box,
              hipStream_t st, int* nblocks);

// ---- many sets in one launch (vpm_batch_run_rows) ----
struct Row32Batch {
  const int* set_off;     // [S + 1]
  const int* item_set;    // [items]
  const int* item_block;  // [items] target block of rows_per_item rows
  int nsets, n_items, rows_per_item, splits;
  int* chunk0;            // [S + 1] filled here
  float* rec;
  double* box;
};

// Source splits of every row for these items, and the bytes they take.
int row32_batch_splits(int64_t n, int n_items, int rows_per_item);
size_t row32_batch_split_bytes(int64_t n, int splits);
size_t row32_batch_record_bytes(int64_t n, int nsets);
size_t row32_batch_box_bytes(int64_t n, int nsets);

// a: outputs, src, perm, n (all sets'), ens_part with n_items * rows_per_item
// slots, part (b.splits > 1).  mask: 3, 7, 27 or 31.
int row32_batch_run(const FusedArgs& a, const Row32Batch& b, unsigned mask, hipStream_t st);

}  // namespace vpm
