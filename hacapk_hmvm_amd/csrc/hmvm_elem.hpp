// hmvm_elem.hpp -- element types of slots and multi-RHS vectors and their
// vector loads and stores (device code shared by the kernels).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace hmvm {

// Element type of the slot buffers (per-tile sums): the tile's accumulation
// type.  A lane-per-row tile's FP32 sum is stored exactly; a column-split
// tile adds its groups' FP32 partials in FP64 and stores that sum rounded
// once to FP32.  The segment sums that add slots into t and y accumulate in
// FP64.  FP32 and BF16 storage thus move half the slot bytes of FP64.  (The
// slots of the multi-RHS groups are FP64 in all storages.)
template <typename S>
struct SlotOf { using T = float; };
template <>
struct SlotOf<double> { using T = double; };

// Element type of the multi-RHS vectors the tiles read (the copy of X and
// t): the MFMA operand type, i.e. FP64, FP32, and for BF16 storage the BF16
// bits of the FP32-rounded value (round to nearest even twice, as the
// operand conversion of the FP32 value would do).
template <typename S>
struct VecOf { using T = S; };

__device__ __forceinline__ short bf16_bits(float f) {
  const uint32_t b = __float_as_uint(f);
  return (short)(uint16_t)((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
}

// NB consecutive elements at p (p aligned to NB elements): one 4-, 8- or
// 16-byte access per 16 bytes.
__device__ __forceinline__ double from_bf16(uint32_t b) { return (double)__uint_as_float(b << 16); }
__device__ __forceinline__ uint32_t to_bf16(double v) { return (uint32_t)(uint16_t)bf16_bits((float)v); }

template <int NB, typename T>
__device__ __forceinline__ void load_n(const T *__restrict__ p, double (&v)[NB]) {
  if constexpr (std::is_same<T, uint16_t>::value) {  // BF16 bits
    if constexpr (NB == 1) {
      v[0] = from_bf16(p[0]);
    } else if constexpr (NB == 2) {
      const uint32_t w = *reinterpret_cast<const uint32_t *>(p);
      v[0] = from_bf16(w & 0xFFFFu);
      v[1] = from_bf16(w >> 16);
    } else {
#pragma unroll
      for (int c = 0; c < NB; c += 4) {
        const uint2 w = *reinterpret_cast<const uint2 *>(p + c);
        v[c] = from_bf16(w.x & 0xFFFFu);
        v[c + 1] = from_bf16(w.x >> 16);
        v[c + 2] = from_bf16(w.y & 0xFFFFu);
        v[c + 3] = from_bf16(w.y >> 16);
      }
    }
  } else if constexpr (NB == 1) {
    v[0] = (double)p[0];
  } else if constexpr (sizeof(T) == 8) {
#pragma unroll
    for (int c = 0; c < NB; c += 2) {
      const double2 w = *reinterpret_cast<const double2 *>(p + c);
      v[c] = w.x;
      v[c + 1] = w.y;
    }
  } else if constexpr (NB == 2) {
    const float2 w = *reinterpret_cast<const float2 *>(p);
    v[0] = (double)w.x;
    v[1] = (double)w.y;
  } else {
#pragma unroll
    for (int c = 0; c < NB; c += 4) {
      const float4 w = *reinterpret_cast<const float4 *>(p + c);
      v[c] = (double)w.x;
      v[c + 1] = (double)w.y;
      v[c + 2] = (double)w.z;
      v[c + 3] = (double)w.w;
    }
  }
}
template <int NB, typename T>
__device__ __forceinline__ void store_n(T *__restrict__ p, const double (&v)[NB]) {
  if constexpr (std::is_same<T, uint16_t>::value) {  // BF16 bits
    if constexpr (NB == 1) {
      p[0] = (uint16_t)to_bf16(v[0]);
    } else if constexpr (NB == 2) {
      *reinterpret_cast<uint32_t *>(p) = to_bf16(v[0]) | (to_bf16(v[1]) << 16);
    } else {
#pragma unroll
      for (int c = 0; c < NB; c += 4)
        *reinterpret_cast<uint2 *>(p + c) =
            uint2{to_bf16(v[c]) | (to_bf16(v[c + 1]) << 16), to_bf16(v[c + 2]) | (to_bf16(v[c + 3]) << 16)};
    }
  } else if constexpr (NB == 1) {
    p[0] = (T)v[0];
  } else if constexpr (sizeof(T) == 8) {
#pragma unroll
    for (int c = 0; c < NB; c += 2) *reinterpret_cast<double2 *>(p + c) = double2{v[c], v[c + 1]};
  } else if constexpr (NB == 2) {
    *reinterpret_cast<float2 *>(p) = float2{(float)v[0], (float)v[1]};
  } else {
#pragma unroll
    for (int c = 0; c < NB; c += 4)
      *reinterpret_cast<float4 *>(p + c) = float4{(float)v[c], (float)v[c + 1], (float)v[c + 2], (float)v[c + 3]};
  }
}

}  // namespace hmvm
