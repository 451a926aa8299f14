// hmvm_stage.hpp -- a plan's stream and its pinned host memory, for the calls
// that take and return host vectors.
//
// hipMemcpyAsync between the device and pageable memory costs a call on host
// vectors 11 to 30 us per vector of 1,000 to 20,000 rows.  Here the CPU copies
// them to or from pinned memory (80 KB: 0.7 us), which one kernel reads into
// device memory and the last kernel of the call writes; the caller
// synchronises once.
#pragma once

#include <hip/hip_runtime.h>

#include "hmvm_hip.h"

namespace hmvm {

constexpr int kStageTail = 16;  // doubles after the two vectors

hipStream_t plan_stream(hmvm_plan *plan);
// 2*nd + kStageTail doubles of pinned memory, made at the first call and kept
// with the plan; nullptr for plans of more than kStageRows rows, or where the
// memory cannot be had.  One call at a time uses it: those that do hold the
// plan's stream until they return.
double *plan_stage(hmvm_plan *plan);
// dst[i] = src[i], n doubles, 16-byte aligned; either side may be pinned.
void stage_copy(double *dst, const double *src, size_t n, hipStream_t st);

}  // namespace hmvm
