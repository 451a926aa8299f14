// hmvm_multi_args.hpp -- arguments and launches of the multi-RHS kernels
// (hmvm_multi.hip), for the runtime.
#pragma once

#include <hip/hip_runtime.h>

#include "hmvm_multi_plan.hpp"

namespace hmvm {

// A row of a vector (64 doubles), or one slice's words of a lane's rows.
constexpr size_t kMultiZeroBytes = 4096;

struct MultiArgs {
  const MultiGroup *__restrict__ groups;
  const MultiWave *__restrict__ waves;
  const MultiItem *__restrict__ items;
  const MultiSlice *__restrict__ slices;
  const void *__restrict__ vals;  // packed values
  const void *__restrict__ X;
  const void *T;             // t (written by launch A, read by launch B)
  const void *__restrict__ zero;  // kMultiZeroBytes of zeros: what columns and batches past the last one read
  double *slots;
  void *t_out;
  const int32_t *__restrict__ tmap;
  const double *__restrict__ mscale;  // BF16: both factor scales of every tmap row's leaf
  double *Y;
  const int2 *__restrict__ yrng;
  const int32_t *__restrict__ ylist;
  int accumulate;
  int y16;  // Y is 16-byte aligned
};

// One workgroup of `waves` waves per group; nrhs 16, 32 or 64; which: 0 the
// stage-1 groups, 1 the rows of y.
void launch_multi_groups(int storage, int nrhs, int which, const MultiArgs &a, int ngroups, int waves, hipStream_t st);
// Packs n records' values (out: MultiPlan::nvals elements of the storage type).
void launch_multi_pack(int storage, int n, const MultiPack *recs, const void *vals, const float *scales, void *out,
                       hipStream_t st);

}  // namespace hmvm
