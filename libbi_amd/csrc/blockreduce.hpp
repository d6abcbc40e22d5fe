// Deterministic wavefront/block reductions (fixed association order).
#pragma once

#include <type_traits>

#include "common.hpp"

namespace bihip {

// op(v, the value of lane ^ O), for a symmetric op: DPP within a row of 16
// lanes, the row and half swaps beyond (a swap of two copies leaves one of the
// pair in each, in both lanes).  No LDS traffic: a shuffle through LDS costs
// its latency in each of the six dependent steps.
template <int O, class Op>
__device__ __forceinline__ double xor_step(double v, Op op) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32, "power of two");
  if constexpr (O == 1) {
    return op(v, dpp<0xB1>(v));  // quad_perm 1,0,3,2
  } else if constexpr (O == 2) {
    return op(v, dpp<0x4E>(v));  // quad_perm 2,3,0,1
  } else if constexpr (O == 4) {
    return op(v, dpp<0x1B>(dpp<0x141>(v)));  // mirrored in eight, then in four
  } else if constexpr (O == 8) {
    return op(v, dpp<0x128>(v));  // row_ror 8
  } else {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
    if constexpr (O == 16) {
      const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
      const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
      return op(__longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0])),
                __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1])));
    } else {
      const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
      const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
      return op(__longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0])),
                __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1])));
    }
  }
}

template <int FROM, class Op>
__device__ __forceinline__ double wave_butterfly(double v, Op op) {
  if constexpr (FROM <= 1) v = xor_step<1>(v, op);
  if constexpr (FROM <= 2) v = xor_step<2>(v, op);
  if constexpr (FROM <= 4) v = xor_step<4>(v, op);
  if constexpr (FROM <= 8) v = xor_step<8>(v, op);
  if constexpr (FROM <= 16) v = xor_step<16>(v, op);
  return xor_step<32>(v, op);
}

// Butterfly reductions over the wave.  FROM > 1: only lanes that are
// multiples of FROM hold values (the others hold the reduction's identity),
// so the exchanges below FROM are skipped; lane 0 and every lane that holds
// a value end with the same result as the full butterfly.
template <int FROM = 1>
__device__ __forceinline__ double wave_max(double v) {
  return wave_butterfly<FROM>(v, [](double a, double b) { return nan_max(a, b); });
}

template <class T, int FROM = 1>
__device__ __forceinline__ T wave_sum(T v) {
  if constexpr (std::is_same<T, double>::value) {
    return wave_butterfly<FROM>(v, [](double a, double b) { return a + b; });
  } else {
#pragma unroll
    for (int o = FROM; o < WAVE; o <<= 1) v += __shfl_xor(v, o, WAVE);
    return v;
  }
}

// Block-wide max (NaN below all); every thread gets the result.
template <int BLOCK, int FROM = 1>
__device__ __forceinline__ double block_max(double v, double* lds) {
  constexpr int NW = BLOCK / WAVE;
  v = wave_max<FROM>(v);
  const int w = threadIdx.x / WAVE, l = threadIdx.x & (WAVE - 1);
  __syncthreads();
  if (l == 0) lds[w] = v;
  __syncthreads();
  double r = lds[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) r = nan_max(r, lds[i]);
  return r;
}

// Block-wide sum; every thread gets the result.
template <int BLOCK, class T, int FROM = 1>
__device__ __forceinline__ T block_sum(T v, T* lds) {
  constexpr int NW = BLOCK / WAVE;
  v = wave_sum<T, FROM>(v);
  const int w = threadIdx.x / WAVE, l = threadIdx.x & (WAVE - 1);
  __syncthreads();
  if (l == 0) lds[w] = v;
  __syncthreads();
  T r = lds[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) r += lds[i];
  return r;
}

// (max, sum exp(lw - max), sum exp(2(lw - max))) over the block's values;
// NaN values (also used for "no value") weigh zero, as bi::nanexp does.
// FROM: values only in lanes that are multiples of FROM (one per lane group).
template <int BLOCK, int FROM = 1>
__device__ __forceinline__ void block_weight_partial(double lw, double* out) {
  __shared__ double lds[BLOCK / WAVE];
  const double m = block_max<BLOCK, FROM>(lw, lds);
  const double z = nanexp(lw - m);
  const double s1 = block_sum<BLOCK, double, FROM>(z, lds);
  const double s2 = block_sum<BLOCK, double, FROM>(z * z, lds);
  if (threadIdx.x == 0) {
    out[0] = m;
    out[1] = s1;
    out[2] = s2;
  }
}

}  // namespace bihip
