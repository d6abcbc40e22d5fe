// Device helpers of the BF16 MFMA multilayer perceptron (mlp.hip, surrogate.hip).
//
// bfloat16 values live in memory as uint16_t and reach the matrix cores as
// 8-element vectors.  The operand layouts of v_mfma_f32_32x32x16_bf16 on
// gfx950 (64 lanes, 16 FP32 accumulators per lane):
//   A (32 x 16): lane l holds A[l % 32][8 (l / 32) + j], j = 0..7
//   B (16 x 32): lane l holds B[8 (l / 32) + j][l % 32], j = 0..7
//   C (32 x 32): accumulator r of lane l is C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32]
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bihip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32v4 __attribute__((ext_vector_type(4)));

// float -> bfloat16 in the high half of a word, round to nearest even; a NaN
// stays a NaN (quiet, sign and payload kept).  Branch-free: the NaN case is a
// select, so the fused kernels carry no exec-mask branches per activation.
__device__ __forceinline__ uint32_t f2bf_hi(float f) {
  const uint32_t u = __float_as_uint(f);
  const uint32_t r = u + 0x7fffu + ((u >> 16) & 1u);
  return __builtin_isnan(f) ? (u | 0x400000u) : r;
}

// float -> bfloat16, round to nearest even (NaN stays NaN)
__device__ __forceinline__ uint16_t f2bf(float f) { return (uint16_t)(f2bf_hi(f) >> 16); }

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// two floats -> packed bfloat16 pair (low half = a), round to nearest even:
// the two high halves joined by one byte permute.  (The integer form keeps
// the fused kernels' register allocation free of spills, which the
// compiler's v_cvt_pk_bf16_f32 lowering did not.)
__device__ __forceinline__ uint32_t pack_bf2(float a, float b) {
  return __builtin_amdgcn_perm(f2bf_hi(b), f2bf_hi(a), 0x07060302u);
}

// two floats -> packed bfloat16 pair by the chip's conversion (round to nearest
// even, as pack_bf2).  Written out, because the compiler's lowering of the
// conversion spilled in the fused kernels.  The matrix instructions that read
// the result come after the workgroup barrier that ends the layer; volatile
// keeps it on this side of that barrier.
__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  uint32_t r;
  asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// GELU in its sigmoid form z sigma(1.702 z) (Hendrycks & Gimpel 2016, sec. 2):
// one exponential and one reciprocal per activation.  Derivative
// s + 1.702 z s (1 - s) with s = sigma(1.702 z).
__device__ __forceinline__ float gelu_sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-1.702f * z));
}
__device__ __forceinline__ float gelu_f(float z) { return z * gelu_sigmoid(z); }
__device__ __forceinline__ float gelu_grad_f(float z) {
  const float s = gelu_sigmoid(z);
  return s + 1.702f * z * s * (1.0f - s);
}

__device__ __forceinline__ f32x16 mfma32(const u16x8& a, const u16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(const u16x8& a, const u32v4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// row of accumulator r of lane l in a 32 x 32 tile
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// ---------------------------------------------------------------- fused inference
// Layers computed transposed, out^T = W in^T, for 32 particles per wave: the
// weights are the A operand (rows staged in LDS), the activations the B operand
// held in registers as packed bfloat16 pairs (act[c][0..3] = inputs
// 16 c + 8 h + 0..7 of the lane's particle, h = lane / 32).  An output tile's
// accumulator lands in the lane that owns the particle, with the rows of each
// 16-block in the order [0-3, 8-11, 4-7, 12-15] across the two half-waves;
// layers fed by such outputs store their input columns in that order (the
// inference weights).
//
// A workgroup's waves walk through the network in chunks of weight rows, two
// LDS buffers in turn: the chunk after the one being computed is copied from
// global memory straight to LDS meanwhile (stage_async), so a chunk costs one
// barrier and no exposed load.  The copy writes runs of 1 KB, 64 pieces of 16
// bytes, one a lane.  Sixteen consecutive rows read the same piece together;
// StagedRows<K> places the pieces so that these 16 lie in different banks, at
// addresses of few registers plus constants:
//   K = 256: two rows a run, the odd one with its piece index XOR 8; runs 16
//            bytes apart;
//   K = 64:  eight rows a run, the piece index XOR (row % 8) / 2; runs 64 bytes
//            apart;
//   K = 320: rows one after another, the low three bits of the piece index XOR
//            (row / 2) % 8.
template <int K>
struct StagedRows;

template <>
struct StagedRows<256> {
  static constexpr int GAP = 16, BASES = 2, TILE = 16 * (1024 + GAP);  // bytes of 32 rows
  static constexpr int bytes(int rows) { return rows / 2 * (1024 + GAP); }
  __device__ __forceinline__ static void piece_of(int slot, int& row, int& piece) {
    row = slot >> 5;
    piece = (slot & 31) ^ ((row & 1) << 3);
  }
  __device__ __forceinline__ static void bases(int row, int h, int (&b)[BASES]) {
    const int at = (row >> 1) * (1024 + GAP) + (row & 1) * 512 + 16 * h;
    b[0] = at + (row & 1) * 128;
    b[1] = at - (row & 1) * 128;
  }
  static constexpr int base(int c) { return (c >> 2) & 1; }
  static constexpr int offset(int c) { return 32 * c; }
};

template <>
struct StagedRows<64> {
  static constexpr int GAP = 64, BASES = 2, TILE = 4 * (1024 + GAP);
  static constexpr int bytes(int rows) { return rows / 8 * (1024 + GAP); }
  __device__ __forceinline__ static void piece_of(int slot, int& row, int& piece) {
    row = slot >> 3;
    piece = (slot & 7) ^ ((row >> 1) & 3);
  }
  __device__ __forceinline__ static void bases(int row, int h, int (&b)[BASES]) {
    const int at = (row >> 3) * (1024 + GAP) + (row & 7) * 128, k = (row >> 1) & 3;
    b[0] = at + 16 * (h ^ k);
    b[1] = at + 16 * ((2 + h) ^ k);
  }
  static constexpr int base(int c) { return c & 1; }
  static constexpr int offset(int c) { return 64 * (c >> 1); }
};

template <>
struct StagedRows<320> {
  static constexpr int GAP = 0, BASES = 4, TILE = 32 * 640;
  static constexpr int bytes(int rows) { return rows * 640; }
  __device__ __forceinline__ static void piece_of(int slot, int& row, int& piece) {
    row = slot / 40;
    piece = (slot % 40) ^ ((row >> 1) & 7);
  }
  __device__ __forceinline__ static void bases(int row, int h, int (&b)[BASES]) {
    const int at = row * 640, k = (row >> 1) & 7;
#pragma unroll
    for (int q = 0; q < 4; ++q) b[q] = at + 16 * ((2 * q + h) ^ k);
  }
  static constexpr int base(int c) { return c & 3; }
  static constexpr int offset(int c) { return 128 * (c >> 2); }
};

// Starts the copy of rows [row0, row0 + NROWS) of a row-major [.][K] bf16
// matrix into `buf`; complete after stage_wait.  Written as instructions: with
// the builtin the compiler waits for the copy before the next LDS read of any
// address, which ends the overlap.  The loads write no register; they are
// counted in vmcnt, so a wait of the compiler's own can only come late because
// of them, never early.  m0 holds their LDS address.
template <int NROWS, int K, int THREADS>
__device__ __forceinline__ void stage_async(const uint16_t* __restrict__ W, int row0,
                                            uint8_t* buf) {
  using S = StagedRows<K>;
  constexpr int SLOTS = NROWS * (K / 8);
  static_assert(SLOTS % THREADS == 0 && THREADS % 64 == 0, "whole runs for every wave");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)buf;
#pragma unroll
  for (int it = 0; it < SLOTS / THREADS; ++it) {
    const int run = it * (THREADS / 64) + wave;
    int row, piece;
    S::piece_of(64 * run + lane, row, piece);
    const uint16_t* src = W + (size_t)(row0 + row) * K + 8 * piece;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(lds0 + (uint32_t)(run * (1024 + S::GAP))), "v"(src)
                 : "m0", "memory");
  }
}

// This wave's copies are in LDS, every wave's after the barrier, which also ends
// the reads of the buffer that the next stage_async fills.
__device__ __forceinline__ void stage_wait() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// The A operands of 32 rows for this lane: rows from a multiple of 32 of the
// staged chunk, input chunk c of 16.
template <int K>
struct StagedTile {
  using S = StagedRows<K>;
  const uint8_t* b[S::BASES];
  __device__ __forceinline__ StagedTile(const uint8_t* buf, int lane) {
    int at[S::BASES];
    S::bases(lane & 31, lane >> 5, at);
#pragma unroll
    for (int q = 0; q < S::BASES; ++q) b[q] = buf + at[q];
  }
  __device__ __forceinline__ u16x8 operator()(int tile, int c) const {
    return *reinterpret_cast<const u16x8*>(b[S::base(c)] + tile * S::TILE + S::offset(c));
  }
};

// n floats into LDS (the biases), by the whole workgroup
__device__ __forceinline__ void copy_floats(const float* __restrict__ src, int n, float* dst,
                                            int threads) {
  for (int i = threadIdx.x; i < n; i += threads) dst[i] = src[i];
}

// biases (LDS, from row 0) of the accumulators of output tile t
__device__ __forceinline__ f32x16 bias_tile(const float* bias, int t, int lane) {
  f32x16 acc;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 b = *reinterpret_cast<const float4*>(&bias[32 * t + 8 * q + 4 * (lane >> 5)]);
    acc[4 * q] = b.x;
    acc[4 * q + 1] = b.y;
    acc[4 * q + 2] = b.z;
    acc[4 * q + 3] = b.w;
  }
  return acc;
}

// Output tiles [T0, T1) of a GELU layer with KC input chunks: buf holds rows
// from 32 T0 on; out[2 t + s] receives the packed activations of tile t.  (Two
// waves share a SIMD: one's activations run beside the other's matrix
// instructions.  Computing a tile's activations between the next tile's matrix
// instructions of the same wave measured the same on the surrogate flow.)
template <int KC, int NOUTC, int K, int T0, int T1>
__device__ __forceinline__ void gelu_tiles(const uint8_t* buf, const float* bias,
                                           const uint32_t (&in)[KC][4],
                                           uint32_t (&out)[NOUTC][4], int lane) {
  const StagedTile<K> W(buf, lane);
#pragma unroll
  for (int t = T0; t < T1; ++t) {
    const f32x16 b = bias_tile(bias, t, lane);
    f32x16 acc{};
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const u32v4 bv = {in[c][0], in[c][1], in[c][2], in[c][3]};
      acc = mfma32(W(t - T0, c), bv, acc);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      out[2 * t + (q >> 2)][q & 3] = cvt_pk_bf16(gelu_f(acc[2 * q] + b[2 * q]),
                                                 gelu_f(acc[2 * q + 1] + b[2 * q + 1]));
  }
}

// one linear output tile (rows [32 tl, 32 tl + 32) of the staged chunk; biases
// of tile t) of a layer with KC input chunks; BIAS_FIRST: the products are added
// to the bias, else the bias to their sum
template <int KC, int K, bool BIAS_FIRST>
__device__ __forceinline__ f32x16 linear_tile(const uint8_t* buf, int tl, int t,
                                              const float* bias, const uint32_t (&in)[KC][4],
                                              int lane) {
  const StagedTile<K> W(buf, lane);
  const f32x16 b = bias_tile(bias, t, lane);
  f32x16 acc{};
  if constexpr (BIAS_FIRST) acc = b;
#pragma unroll
  for (int c = 0; c < KC; ++c) {
    const u32v4 bv = {in[c][0], in[c][1], in[c][2], in[c][3]};
    acc = mfma32(W(tl, c), bv, acc);
  }
  if constexpr (!BIAS_FIRST) acc += b;
  return acc;
}

}  // namespace bihip
