// hmvm_multi.hpp -- gfx950 kernels of the products with several right-hand
// sides (schedule and packed values: hmvm_multi_plan.hpp).
//
// Y (nd x nrhs, row-major) (+)= A X, nrhs = 16*NB right-hand sides.
//   FP64 storage: v_mfma_f64_16x16x4_f64   (K = 4, FP64 accumulate)
//   FP32 storage: v_mfma_f32_16x16x4_f32   (K = 4, FP32 accumulate)
//   BF16 storage: v_mfma_f32_16x16x32_bf16 (K = 32, vector entries in BF16,
//                 FP32 accumulate; stage 1 v_mfma_f32_16x16x16_bf16)
// Operand layouts (wave64): A lane l holds row l%16 of K-slice l/16, B lane l
// right-hand side l%16 of the same K-slice (one column for K = 4, eight for
// K = 32); the 16x16 result gives lane l four rows of column l%16:
// 4*(l/16)+v for the FP32 and BF16 instructions, l/16+4v for the FP64 one.
// Which column stands at which k is free as long as both operands agree: the
// 16 lanes of K-slice g take the KS consecutive columns of slice g of a
// batch, so a batch is four MFMA steps (FP64, FP32) or one (BF16), and a
// lane's matrix words are its A operands as loaded.  Block cb, MFMA column j
// is right-hand side NB*j + cb, so a lane's NB right-hand sides are one
// vector load.
#pragma once

#include "hmvm_elem.hpp"
#include "hmvm_multi_args.hpp"

namespace hmvm {

typedef double mf_d2 __attribute__((ext_vector_type(2)));
typedef double mf_d4 __attribute__((ext_vector_type(4)));
typedef float mf_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 mf_b8 __attribute__((ext_vector_type(8)));
// X may be 8-byte aligned only; global loads need no more than 4.
typedef double mf_d2u __attribute__((ext_vector_type(2), aligned(8)));

template <typename S>
struct Mfma;
template <>
struct Mfma<double> {
  static constexpr int KS = 4, E = 2, H = 2;
  using Acc = mf_d4;
  using Word = mf_d2;  // 16 bytes of a row: E columns
  __device__ static __forceinline__ int row(int lane, int v) { return (lane >> 4) + 4 * v; }  // (measured on gfx950)
};
template <>
struct Mfma<float> {
  static constexpr int KS = 4, E = 4, H = 1;
  using Acc = mf_f4;
  using Word = mf_f4;
  __device__ static __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};
template <>
struct Mfma<uint16_t> {
  static constexpr int KS = 8, E = 8, H = 1;
  using Acc = mf_f4;
  using Word = mf_b8;
  __device__ static __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

__device__ __forceinline__ mf_d4 mfma_step(double a, double b, mf_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mf_f4 mfma_step(float a, float b, mf_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mf_f4 mfma_step(mf_b8 a, mf_b8 b, mf_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

typedef short mf_s4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ mf_f4 mfma_step16(mf_s4 a, mf_s4 b, mf_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Halves h (0 low, 1 high) of words a and b as one word {a, b}.
__device__ __forceinline__ uint32_t pack_half(uint32_t a, uint32_t b, int h) {
  return __builtin_amdgcn_perm(b, a, h ? 0x07060302u : 0x05040100u);
}
union Bf16x8 {
  uint32_t u[4];
  mf_b8 v;
  mf_s4 h[2];
};

// NB consecutive right-hand sides of a vector row, as loaded.
template <typename V, int NB>
struct RhsWord;
template <int NB>
struct RhsWord<double, NB> {
  double v[NB];
};
template <int NB>
struct RhsWord<float, NB> {
  float v[NB];
};
template <>
struct RhsWord<uint16_t, 1> {
  uint32_t u[1];
};
template <int NB>
struct RhsWord<uint16_t, NB> {
  uint32_t u[NB / 2];
};
// X may be 8-byte aligned only: element-aligned loads.
template <int NB>
__device__ __forceinline__ void load_rhs(const double *__restrict__ p, RhsWord<double, NB> &w) {
  if constexpr (NB == 1) {
    w.v[0] = p[0];
  } else {
#pragma unroll
    for (int c = 0; c < NB; c += 2) {
      const mf_d2u d = *reinterpret_cast<const mf_d2u *>(p + c);
      w.v[c] = d[0];
      w.v[c + 1] = d[1];
    }
  }
}
template <int NB>
__device__ __forceinline__ void load_rhs(const float *__restrict__ p, RhsWord<float, NB> &w) {
  if constexpr (NB == 1) {
    w.v[0] = p[0];
  } else if constexpr (NB == 2) {
    const float2 d = *reinterpret_cast<const float2 *>(p);
    w.v[0] = d.x;
    w.v[1] = d.y;
  } else {
    const float4 d = *reinterpret_cast<const float4 *>(p);
    w.v[0] = d.x;
    w.v[1] = d.y;
    w.v[2] = d.z;
    w.v[3] = d.w;
  }
}
template <int NB>
__device__ __forceinline__ void load_rhs(const uint16_t *__restrict__ p, RhsWord<uint16_t, NB> &w) {
  if constexpr (NB == 1) {
    w.u[0] = p[0];
  } else if constexpr (NB == 2) {
    w.u[0] = *reinterpret_cast<const uint32_t *>(p);
  } else {
    const uint2 d = *reinterpret_cast<const uint2 *>(p);
    w.u[0] = d.x;
    w.u[1] = d.y;
  }
}

// What one batch loads: NT row tiles of 16 rows, KS columns a lane.
template <typename S, int NB, int NT>
struct MultiLoads {
  typename Mfma<S>::Word a[NT][Mfma<S>::H];
  RhsWord<typename VecOf<S>::T, NB> x[Mfma<S>::KS];
  int end;  // kOrdered: the batch ends a chunk
};

// Batches whose loads are in flight at once: two (three and four cost
// registers and instruction cache and were slower, FP64 0.56 -> 0.65 and BF16
// 0.188 -> 0.217 ms at N=101,250 with 32 right-hand sides), one where the sums
// leave no registers for a second (BF16 rows of y, 64 right-hand sides, four
// row tiles: two spill 108 bytes a lane, N=50,021 143 -> 137 us with one).
template <typename S, int NB, int NT, bool kOrdered>
constexpr int multi_depth() {
  return NB == 4 && (sizeof(S) >= 4 || (!kOrdered && NT == 4)) ? 1 : 2;
}
// How a column loop ends when its batches are not a multiple of the depth:
// with a tail (more code), or with batches of zeros read from the zero page
// (more products); N=101,250, 32 right-hand sides, tail / zeros: FP64 0.557 /
// 0.545, FP32 0.331 / 0.354, BF16 0.195 / 0.177 ms; BF16 with 64 at N=50,021
// 0.122 / 0.130.
template <typename S, int NB>
constexpr bool multi_tail() {
  return sizeof(S) == 4 || (sizeof(S) == 2 && NB == 4);
}

// An even share of a group's columns is a longer chain of roundings than a
// tile of the one-vector launches, so the MFMA sums of a few columns are folded
// into FP64 sums.  Error against 80 bits, one chain / folded / the tile
// launches: FP64 (32 right-hand sides) N=12,007 6.9e-16 / 2.4e-16 / 4.0e-16,
// N=101,250 1.02e-15 / 3.3e-16 / 7.1e-16; FP32 N=101,250 5.1e-7 / 1.35e-7 / 3.6e-7,
// 64 right-hand sides 1.0e-7 (1.8e-7 with FP32 sums).  BF16: the operands' 2.2e-3
// in all three, but one chain lost 1,023 ones next to 2^30, and made shares above
// FLT_MAX infinite.
// multi_fold: whether a second set of sums for all MFMA tiles takes multi_depth
// batches, where the registers hold it; else each batch of each tile is folded
// (FP64, 32 right-hand sides: a second set 540 -> 650 us at N=101,250).  Without
// the barriers between the tiles the compiler keeps several sums and spills
// (N=101,250: FP64 32 538 -> 560, 64 830 -> 928; FP32 64 542 -> 593).
// us, one chain / folded: FP64 32 right-hand sides N=12,007 93 / 94, N=101,250
// 535 / 534, 64 146 / 157 and 809 / 838 (each fold waits for its MFMA: 18 cycles);
// FP32 64 119 / 109, 551 / 543 (FP32 sums before); BF16 32 39 / 40, N=50,021 (leaf
// 16) 120 / 127, 64 52 / 52, 164 / 171 (fewer waves beside FP64 sums).
// BF16 stage 1 (kOrdered) folds a chunk at its end.
template <typename S, int NB, int NT, bool kOrdered>
constexpr bool multi_fold() {
  return kOrdered || NB == 1 || (sizeof(S) < 8 && NB == 2) || (sizeof(S) != 4 && NB == 4 && NT <= 2);
}

// out += the item's columns: D batches of loads in flight, and the slices of
// the D after those.  kOrdered (BF16 stage 1): a batch is two steps of 16
// columns, one after the other (ordered_column).
template <typename S, int NB, int NT, bool kOrdered>
__device__ __forceinline__ void multi_columns(const MultiArgs &a, const MultiItem &it, int lane,
                                              mf_d4 (&out)[NT][NB]) {
  using M = Mfma<S>;
  using V = typename VecOf<S>::T;
  constexpr int KS = M::KS, E = M::E, H = M::H, nrhs = 16 * NB;
  const int i = lane & 15, g = lane >> 4, nr = it.nrows, nb = it.nbatch;
  if (nb == 0) return;
  const MultiSlice *sl = a.slices + it.slice0 + g;
  // this lane's rows; lanes past the item's rows load its first rows
  const S *ap = (const S *)a.vals + it.a0 + (int64_t)g * nr * KS;
  int off[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) off[t] = (16 * t + i < nr ? 16 * t + i : i < nr ? i : 0) * E;
  const V *X = (const V *)a.X + NB * i, *T = (const V *)a.T + NB * i, *Z = (const V *)a.zero + NB * i;
  auto load = [&](MultiLoads<S, NB, NT> &l, const MultiSlice s, bool on) {
    const S *av = on ? ap : (const S *)a.zero;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int h = 0; h < H; ++h)
        l.a[t][h] = __builtin_nontemporal_load(reinterpret_cast<const typename M::Word *>(av + h * nr * E + off[t]));
    ap += kMultiBatch * KS * nr;
    const V *xr = ((s.info & kSliceT) ? T : X) + (int64_t)s.v * nrhs;
    l.end = on ? s.info & kSliceEnd : 0;
    const int n = on ? s.info & 15 : 0, n2 = on ? (s.info >> 4) & 15 : 0;
#pragma unroll
    for (int q = 0; q < KS; ++q) {
      if (kOrdered && q == kHalf) xr += (kStep - kHalf) * nrhs;
      const bool in_use = kOrdered && q >= kHalf ? q - kHalf < n2 : q < n;
      load_rhs<NB>(in_use ? xr : Z, l.x[q]);  // the zero columns of a slice meet zeros
      xr += nrhs;
    }
  };
  typename M::Acc part[multi_fold<S, NB, NT, kOrdered>() ? NT : 1][NB];
  auto clear = [&]() {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) part[t][cb] = typename M::Acc{0, 0, 0, 0};
  };
  auto add = [](mf_d4 &o, const typename M::Acc &p) {
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] += p[v];
  };
  auto fold = [&]() {
    if constexpr (multi_fold<S, NB, NT, kOrdered>()) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) add(out[t][cb], part[t][cb]);
      clear();
    }
  };
  if constexpr (multi_fold<S, NB, NT, kOrdered>()) clear();
  auto fold_all = [&]() {  // after D batches, where chunks do not say
    if constexpr (!kOrdered) fold();
  };
  auto products = [&](const MultiLoads<S, NB, NT> &l) {
    if constexpr (sizeof(S) == 2) {
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) {
        Bf16x8 b;
#pragma unroll
        for (int q = 0; q < KS; q += 2) b.u[q / 2] = pack_half(l.x[q].u[cb / 2], l.x[q + 1].u[cb / 2], cb & 1);
        if constexpr (kOrdered) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              Bf16x8 w;
              w.v = l.a[t][0];
              part[t][cb] = mfma_step16(w.h[h], b.h[h], part[t][cb]);
            }
        } else {
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            if constexpr (multi_fold<S, NB, NT, kOrdered>()) {
              part[t][cb] = mfma_step(l.a[t][0], b.v, part[t][cb]);
            } else {
              add(out[t][cb], mfma_step(l.a[t][0], b.v, typename M::Acc{0, 0, 0, 0}));
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
      }
      if constexpr (kOrdered)
        if (__builtin_amdgcn_readfirstlane(l.end)) fold();
    } else if constexpr (multi_fold<S, NB, NT, kOrdered>()) {
#pragma unroll
      for (int q = 0; q < KS; ++q)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int cb = 0; cb < NB; ++cb) part[t][cb] = mfma_step(l.a[t][q / E][q % E], l.x[q].v[cb], part[t][cb]);
    } else {  // one MFMA tile after the other, so that one sum of the batch is live at a time
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          typename M::Acc sum{0, 0, 0, 0};
#pragma unroll
          for (int q = 0; q < KS; ++q) sum = mfma_step(l.a[t][q / E][q % E], l.x[q].v[cb], sum);
          add(out[t][cb], sum);
          __builtin_amdgcn_sched_barrier(0);
        }
    }
  };
  constexpr int D = multi_depth<S, NB, NT, kOrdered>();
  MultiLoads<S, NB, NT> l[D];
  MultiSlice s[D];
#pragma unroll
  for (int d = 0; d < D; ++d) s[d] = sl[kMultiBatch * (d < nb ? d : 0)];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    load(l[d], s[d], d < nb);
    s[d] = sl[kMultiBatch * (D + d < nb ? D + d : 0)];
  }
  // No load in these loops is conditional: a branch around one makes the
  // compiler wait for all loads in flight where its paths meet.
  if constexpr (multi_tail<S, NB>()) {
    int b = 0;
    for (; b + 2 * D <= nb; b += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        products(l[d]);
        load(l[d], s[d], true);
        s[d] = sl[kMultiBatch * (b + d + 2 * D < nb ? b + d + 2 * D : 0)];
      }
      fold_all();
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (b + d < nb) products(l[d]);
      if (b + d + D < nb) load(l[d], s[d], true);
    }
    fold_all();
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (b + d + D < nb) products(l[d]);
    fold_all();
  } else {
    for (int b = 0; b < nb; b += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        products(l[d]);
        load(l[d], s[d], b + d + D < nb);
        s[d] = sl[kMultiBatch * (b + d + 2 * D < nb ? b + d + 2 * D : 0)];
      }
      fold_all();
    }
  }
}

// MFMA tiles whose sums of all waves are added at once: 8 KiB of LDS a wave.
// LDS words and slots are FP64 in all storages: a wave's share of a group's
// columns may add up to more than FLT_MAX where the rows of y, or t scaled by
// its leaf's factors, are finite numbers.
template <int NB>
constexpr int multi_piece() {
  return 4 / NB;
}
constexpr int kMultiLdsWave = 8192;  // bytes

// W right-hand sides c.. of the t row that entry m of the row map names
// (BF16: times both factor scales of its leaf).
template <typename S, int NB, int W>
__device__ __forceinline__ void store_t(const MultiArgs &a, int m, int c, double (&r)[W]) {
  const int e = a.tmap[m];
  if constexpr (sizeof(S) == 2) {
    const double f = a.mscale[m];
#pragma unroll
    for (int k = 0; k < W; ++k) r[k] *= f;
  }
  store_n<W>((typename VecOf<S>::T *)a.t_out + (int64_t)e * (16 * NB) + c, r);
}

// One item of NT row tiles: a partial one's rows go to its slots; the kept
// one's are added over the waves (in wave order, FP64) and go to y, t or a
// t slot.
template <typename S, int NB, int NT, bool kOrdered>
__device__ __forceinline__ void multi_item(const MultiArgs &a, const MultiGroup &grp, const MultiItem &it, int lane,
                                           double *lds) {
  using M = Mfma<S>;
  constexpr int nrhs = 16 * NB;
  constexpr int PT = multi_piece<NB>() < NT ? multi_piece<NB>() : NT;
  constexpr int W = 4;  // right-hand sides a thread adds: with two, twice the rounds of dependent slot loads (BF16,
                        // 64 right-hand sides, N=50,021: 174 -> 163 us a product)
  mf_d4 acc[NT][NB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) acc[t][cb] = mf_d4{0, 0, 0, 0};
  multi_columns<S, NB, NT, kOrdered>(a, it, lane, acc);
  if (it.kind != kItemKept) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * t + M::row(lane, v);
        if (row >= it.nrows) continue;
        double r[NB];
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) r[cb] = acc[t][cb][v];
        if (it.kind == kItemSlot)
          store_n<NB>(a.slots + ((int64_t)it.out + row) * nrhs + NB * (lane & 15), r);
        else
          store_t<S, NB>(a, it.out + row, NB * (lane & 15), r);
      }
    return;
  }
  const int nthreads = (int)blockDim.x, nw = nthreads >> 6, w = (int)(threadIdx.x >> 6);
  double *mine = lds + w * PT * 256 * NB;
#pragma unroll
  for (int t0 = 0; t0 < NT; t0 += PT) {
    __syncthreads();  // the previous piece is read, and this workgroup's slots are written
#pragma unroll
    for (int t = t0; t < t0 + PT && t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        double r[NB];
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) r[cb] = acc[t][cb][v];
        store_n<NB>(mine + ((t - t0) * 16 + M::row(lane, v)) * nrhs + NB * (lane & 15), r);
      }
    __syncthreads();
    const int nt = NT - t0 < PT ? NT - t0 : PT;
    for (int e = (int)threadIdx.x; e < nt * 16 * nrhs / W; e += nthreads) {
      const int c = e * W % nrhs, ri = e * W / nrhs;  // right-hand sides c.., tile row ri
      const int row = 16 * t0 + ri;
      if (row >= grp.nrows) continue;
      double s[W];
#pragma unroll
      for (int k = 0; k < W; ++k) s[k] = 0;
      for (int q = 0; q < nw; ++q) {
        double r[W];
        load_n<W>(lds + (q * PT * 16 + ri) * nrhs + c, r);
#pragma unroll
        for (int k = 0; k < W; ++k) s[k] += r[k];
      }
      if (grp.kind == kMultiY) {
        const int64_t y = (int64_t)grp.out + row;
        const int2 rg = a.yrng[y];
        for (int l = rg.x; l < rg.y; ++l) {
          double r[W];
          load_n<W>(a.slots + (a.ylist[l] + y) * nrhs + c, r);
#pragma unroll
          for (int k = 0; k < W; ++k) s[k] += r[k];
        }
        double *o = a.Y + y * nrhs + c;
        if (a.y16) {
          if (a.accumulate) {
            double r[W];
            load_n<W>(o, r);
#pragma unroll
            for (int k = 0; k < W; ++k) s[k] = r[k] + s[k];
          }
          store_n<W>(o, s);
        } else {
#pragma unroll
          for (int k = 0; k < W; ++k) o[k] = a.accumulate ? o[k] + s[k] : s[k];
        }
      } else if (grp.kind == kMultiT) {
        store_t<S, NB>(a, grp.out + row, c, s);
      } else {
        store_n<W>(a.slots + ((int64_t)grp.out + row) * nrhs + c, s);
      }
    }
  }
}

// multi_item for the row tiles that `rows` rows take.
template <typename S, int NB, bool kOrdered>
__device__ __forceinline__ void multi_item_rows(const MultiArgs &a, const MultiGroup &grp, const MultiItem &it,
                                                int lane, double *lds) {
  static_assert(kMultiRows <= 64 && kOrderedRows <= 32, "row tiles");
  if (it.nrows <= 16)
    multi_item<S, NB, 1, kOrdered>(a, grp, it, lane, lds);
  else if (kOrdered || it.nrows <= 32)
    multi_item<S, NB, 2, kOrdered>(a, grp, it, lane, lds);
  else if (it.nrows <= 48)
    multi_item<S, NB, 3, kOrdered>(a, grp, it, lane, lds);
  else
    multi_item<S, NB, 4, kOrdered>(a, grp, it, lane, lds);
}

template <typename S, int NB, bool kOrdered>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void multi_kernel(MultiArgs a) {
  extern __shared__ double multi_lds[];
  const int lane = (int)(threadIdx.x & 63);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const MultiGroup grp = a.groups[blockIdx.x];
  const MultiWave wv = a.waves[(int)blockIdx.x * (int)(blockDim.x >> 6) + w];
  for (int i = 0; i < wv.nitems; ++i)
    multi_item_rows<S, NB, kOrdered>(a, grp, a.items[wv.item0 + i], lane, multi_lds);
}

// Packs the values of one record per workgroup (MultiPack); one thread a row
// of a slice, rows across the lanes on both sides.
template <typename S>
__global__ __launch_bounds__(256) void multi_pack_kernel(const MultiPack *__restrict__ recs, const S *__restrict__ vals,
                                                         const float *__restrict__ scales, S *__restrict__ out) {
  using M = Mfma<S>;
  constexpr int KS = M::KS, E = M::E, H = M::H;
  const MultiPack r = recs[blockIdx.x];
  const int nsl = (r.cols + KS - 1) / KS + r.pad;
  float scale = 1.0f;
  if constexpr (sizeof(S) == 2)
    if (r.factor >= 0) scale = scales[r.factor];
  for (int k = (int)threadIdx.x; k < nsl * r.rows; k += (int)blockDim.x) {
    const int s = k / r.rows, row = k - s * r.rows;
    const S *src = vals + r.src + row;
    S v[KS];
#pragma unroll
    for (int q = 0; q < KS; ++q) {
      const int c = r.ordered ? ordered_column(s, q) : s * KS + q;
      v[q] = c < r.cols ? src[(int64_t)c * r.ld] : S(0);
    }
    if constexpr (sizeof(S) == 2)  // a power of two: exact
#pragma unroll
      for (int q = 0; q < KS; ++q) v[q] = (S)(__float_as_uint(__uint_as_float((uint32_t)v[q] << 16) * scale) >> 16);
    S *dst = out + r.dst + (int64_t)s * r.nrows * KS + (int64_t)(r.row0 + row) * E;
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int e = 0; e < E; ++e) dst[(int64_t)h * r.nrows * E + e] = v[h * E + e];
  }
}

}  // namespace hmvm
