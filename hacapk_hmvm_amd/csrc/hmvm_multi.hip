// hmvm_multi.hip -- launches of the multi-RHS group kernels (hmvm_multi.hpp).
#include "hmvm_multi.hpp"

namespace hmvm {

namespace {
template <typename S, int NB, bool kOrdered>
void launch(const MultiArgs &a, int ngroups, int waves, hipStream_t st) {
  hipLaunchKernelGGL((multi_kernel<S, NB, kOrdered>), dim3(ngroups), dim3(64 * waves), (size_t)kMultiLdsWave * waves, st, a);
}
template <typename S, bool kOrdered>
void launch_nb(int nrhs, const MultiArgs &a, int ngroups, int waves, hipStream_t st) {
  if (nrhs == 16)
    launch<S, 1, kOrdered>(a, ngroups, waves, st);
  else if (nrhs == 32)
    launch<S, 2, kOrdered>(a, ngroups, waves, st);
  else
    launch<S, 4, kOrdered>(a, ngroups, waves, st);
}
}  // namespace

void launch_multi_groups(int storage, int nrhs, int which, const MultiArgs &a, int ngroups, int waves, hipStream_t st) {
  if (ngroups == 0) return;
  if (storage == kF64)
    launch_nb<double, false>(nrhs, a, ngroups, waves, st);
  else if (storage == kF32)
    launch_nb<float, false>(nrhs, a, ngroups, waves, st);
  else if (which == 0)
    launch_nb<uint16_t, true>(nrhs, a, ngroups, waves, st);
  else
    launch_nb<uint16_t, false>(nrhs, a, ngroups, waves, st);
}

void launch_multi_pack(int storage, int n, const MultiPack *recs, const void *vals, const float *scales, void *out,
                       hipStream_t st) {
  if (n == 0) return;
  if (storage == kF64)
    hipLaunchKernelGGL((multi_pack_kernel<double>), dim3(n), dim3(256), 0, st, recs, (const double *)vals, scales,
                       (double *)out);
  else if (storage == kF32)
    hipLaunchKernelGGL((multi_pack_kernel<float>), dim3(n), dim3(256), 0, st, recs, (const float *)vals, scales,
                       (float *)out);
  else
    hipLaunchKernelGGL((multi_pack_kernel<uint16_t>), dim3(n), dim3(256), 0, st, recs, (const uint16_t *)vals, scales,
                       (uint16_t *)out);
}

}  // namespace hmvm
