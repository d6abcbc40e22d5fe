// Resampling of one filter by one workgroup, and the offspring expressions and
// the scan it shares with the tiled chain (resample.hip) and the batched step
// (batch.hip).
//
// Replaces (ON_DEVICE): see resample.hip.
#pragma once

#include "scan.hpp"

namespace bihip {

// O_i = min(n, (int)(Ws_i / W * n + a)) with every operation rounded as
// written (SystematicResampler.hpp:47-50).
__device__ __forceinline__ int systematic_offspring(double Ws, double W, int n, double a) {
#pragma clang fp contract(off)
  const double v = Ws / W * (double)n + a;
  const int o = (int)v;
  return o < n ? o : n;
}

// StratifiedResamplerHost.hpp:68-71
__device__ __forceinline__ double stratified_reach(double Ws, double W, int n) {
#pragma clang fp contract(off)
  return Ws / W * (double)n;
}

__device__ __forceinline__ int stratified_offspring(double reach, double alpha, int n) {
#pragma clang fp contract(off)
  const int o = (int)(reach + alpha);
  return o < n ? o : n;
}

// The cumulative offspring with the stratum's keyed uniform.
__device__ __forceinline__ int stratified_keyed(double Ws, double W, int n, uint64_t seed,
                                                uint32_t step, uint32_t batch) {
  const double reach = stratified_reach(Ws, W, n);
  int k = (int)reach;
  if (k > n - 1) k = n - 1;
  const u32x4 r = philox_block(seed, (uint32_t)k, step, TAG_STRATIFIED, batch, 0);
  return stratified_offspring(reach, u53(r.x, r.y), n);
}

// (e, f) = (max(o - 1, 0), [o == 0]) packed as e | f << 32.
__device__ __forceinline__ uint64_t ef_pair(int o) {
  const uint64_t e = o > 1 ? (uint64_t)(o - 1) : 0u;
  const uint64_t f = o == 0 ? 1u : 0u;
  return e | (f << 32);
}

constexpr int SMALL_BLOCK = 1024;

// Inclusive scan of one integer value per thread over the workgroup (at most
// 16 waves); total receives the sum.  Each wave scans the waves' sums in one
// row of lanes; through shuffles and a serial pass over the 16 sums in every
// thread the two scans of the chain took about half of its 7 us.
template <class V>
__device__ __forceinline__ V small_inclusive_scan(V v, V* lds, V& total) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  const int nw = (int)blockDim.x / WAVE;
  v = wave_inclusive_scan(v);
  if (lane == WAVE - 1) lds[w] = v;
  __syncthreads();
  const int q = lane & 15;
  const V s = row_inclusive_scan(q < nw ? lds[q] : V(0));
  total = read_lane(s, 15);
  return w > 0 ? read_lane(s, w - 1) + v : v;
}

// LDS of the chain for N = SMALL_BLOCK * ITEMS particles (MULTINOMIAL: with the
// cumulative weights and the offspring counts).
template <int ITEMS, bool MULTINOMIAL>
struct SmallChainLds {
  static constexpr int N = SMALL_BLOCK * ITEMS;
  u128 l128[SMALL_BLOCK / WAVE];
  uint64_t l64[SMALL_BLOCK / WAVE];
  uint16_t E[N];
  double Ws[MULTINOMIAL ? N : 1];
  int count[MULTINOMIAL ? N : 1];
};

// Ancestors src of the thread's ITEMS consecutive particles (from
// threadIdx.x * ITEMS; blockDim.x * ITEMS >= P) of a filter of P particles with
// log-weights lw and maximum m, n = P draws of step `step`; false (for the whole workgroup) if the
// weights sum to no positive number.  Exact integer sums and the tiled chain's
// expressions, so its ancestors.  Ends with reads of the LDS.
template <int MODE, int ITEMS, class Lds>
__device__ __forceinline__ bool small_chain(const double (&lw)[ITEMS], double m, int P, int n,
                                            uint64_t seed, uint32_t step, uint32_t batch, Lds& L,
                                            int (&src)[ITEMS]) {
  const int base = (int)threadIdx.x * ITEMS;
  // inclusive fixed-point weight sums
  u128 v[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
    v[i] = base + i < P ? fix_weight(nanexp(lw[i] - m)) : u128(0);
#pragma unroll
  for (int i = 1; i < ITEMS; ++i) v[i] = v[i - 1] + v[i];
  u128 tot;
  const u128 start = small_inclusive_scan(v[ITEMS - 1], L.l128, tot) - v[ITEMS - 1];
  const double W = fix_to_double(tot);
  if (!(W > 0.0)) return false;

  // offspring counts
  int o[ITEMS];
  if constexpr (MODE == BIHIP_MULTINOMIAL) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      L.Ws[base + i] = fix_to_double(start + v[i]);
      L.count[base + i] = 0;
    }
    __syncthreads();
    for (int j = threadIdx.x; j < n; j += (int)blockDim.x) {
      const u32x4 r = philox_block(seed, (uint32_t)j, step, TAG_MULTINOMIAL, batch, 0);
      const double u = W * u53(r.x, r.y);
      int lo = 0, hi = P;  // first i with Ws_i > u
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (L.Ws[mid] <= u) lo = mid + 1;
        else hi = mid;
      }
      atomicAdd(&L.count[lo < P ? lo : P - 1], 1);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) o[i] = base + i < P ? L.count[base + i] : 1;
  } else {
    double av = 0.0;
    if (MODE == BIHIP_SYSTEMATIC) {
      const u32x4 r = philox_block(seed, 0, step, TAG_SYSTEMATIC, batch, 0);
      av = u53(r.x, r.y);
    }
    auto cumulative = [&](const u128& incl) -> int {
      const double Wsi = fix_to_double(incl);
      if (MODE == BIHIP_SYSTEMATIC) return systematic_offspring(Wsi, W, n, av);
      return stratified_keyed(Wsi, W, n, seed, step, batch);
    };
    int prev = base > 0 && base < P ? cumulative(start) : 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      o[i] = 1;  // past the end: no extras, not free
      if (base + i < P) {
        const int O = cumulative(start + v[i]);
        o[i] = O - prev;
        prev = O;
      }
    }
  }

  // exclusive sums of extra copies (E) and free slots
  uint64_t t = 0;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) t += ef_pair(o[i]);
  uint64_t eftot;
  uint64_t run = small_inclusive_scan(t, L.l64, eftot) - t;
  int rank[ITEMS];  // of a free slot; -1: occupied
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    L.E[base + i] = (uint16_t)run;
    rank[i] = o[i] == 0 ? (int)(run >> 32) : -1;
    run += ef_pair(o[i]);
  }
  __syncthreads();

  // the free slot of rank r receives the last i with E_i <= r
  int pos[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) pos[i] = 0;  // E_0 = 0
  for (int s = 1 << (31 - __clz(P)); s > 0; s >>= 1) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int c = pos[i] + s;
      if (c < P && (int)L.E[c] <= rank[i]) pos[i] = c;
    }
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
    src[i] = rank[i] < 0 ? base + i : pos[i];
  return true;
}

}  // namespace bihip
