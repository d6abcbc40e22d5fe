// Learned guided proposal for the Lorenz-96 d=200 filter, with the importance
// weight corrected exactly.
//
// The filter step runs the exact flow Phi(x) first (k_transition without
// noise or correction, gathered through the ancestors), then this kernel
// proposes, in place over Phi,
//   x' = Phi + q (m + e^{s/2} eps),   eps ~ N(0, I) (the transition-noise stream),
// where (m, s) = MLP(u) per dimension, u = ((Phi - shift) / scale,
// (y - H Phi) / obs_sd, (F - F0) / F_scale), and adds to the log-weight
//   log p(y | x') + log N(x'; Phi, q^2 I) - log N(x'; Phi + q m, q^2 e^s)
//   = log p(y | x') + sum_i [ -(m_i + e^{s_i/2} eps_i)^2 / 2 + eps_i^2 / 2 + s_i / 2 ].
// With m = 0 and s = 0 it is the bootstrap filter's step, draw for draw.
// The reference's nearest pattern is the auxiliary-weight correction of
// BridgePF / LookaheadPF (share/src/bi/filter/BridgePF.hpp:114-144,
// share/src/bi/filter/LookaheadPF.hpp:91-124); the learned proposal itself
// has no counterpart there.
//
// Network 301-256-256-256-400 (outputs: m for 200 dimensions, then s), BF16
// MFMA with FP32 accumulation, laid out as the surrogate kernel's (32
// particles per wave, weights staged in LDS in row chunks that are copied
// while the chunk before is computed, activations in registers).  2^17
// particles take 0.157 ms (518 TFLOP/s); with every state of the output read
// behind the store before it and the chunks loaded between barriers, 0.233 ms.
// Bound by vector work beside the matrix cores (10600 vector and 624 matrix
// instructions a wave, 37% of the wave cycles waiting) at two waves per SIMD.
// The inference weights of the output layer interleave the rows per 16
// dimensions (m of dimensions 16 t .. 16 t + 15, then their s), so one 32-row
// output tile carries both numbers of the dimensions it covers.
#include <type_traits>

#include "blockreduce.hpp"
#include "internal.hpp"
#include "mlp.hpp"
#include "model_ops.hpp"

namespace bihip {

struct GuidedArgs {
  const uint16_t* W[MLP_MAX_LAYERS];
  const float* b[MLP_MAX_LAYERS];
  float x_shift, x_inv_scale, innov_inv, par_u;
  float* X;          // in: Phi, out: x' (column-major, ld)
  int ld, P;
  const double* y;   // observations of this step (filter mode: from dev)
  uint64_t seed;
  uint32_t batch, step;
  float q;           // transition noise sd
  double obs_sd;
  // filter mode
  const PFDevice* dev;
  const double* y_base;
  int nobs;
  double* lws;
  double* partials;
  // standalone mode: log-weight increment per particle
  double* inc;
  const int* imp_r;  // filter mode: imposed resampling flags per step (nullable)
  BankStrides bk;    // filter mode: filter blockIdx.y of a bank at these strides
  const float* par_u_bank;  // bank: the parameter input per filter (nullable)
};

namespace {

constexpr int GP_THREADS = 512, GP_TILE = 256;
constexpr int GD = 200, GNOBS = 100, GH = 256;
constexpr int GK0 = 320;                 // 301 inputs padded
constexpr int GOUT_TILES = (GD + 15) / 16;  // 13 tiles of 16 dimensions (m and s)
constexpr int GHR = GH / 2;              // rows of a chunk of a hidden layer
constexpr int G0R = 64;                  // rows of a chunk of layer 0

template <bool FILTER>
__global__ __launch_bounds__(GP_THREADS) void k_guided(GuidedArgs a) {
  // two chunks of weights (stage_async) and the biases: 128 KB + 4.7 KB
  static_assert(StagedRows<GK0>::bytes(G0R) <= StagedRows<GH>::bytes(GHR), "chunks of layer 0");
  __shared__ __attribute__((aligned(16))) uint8_t buf[2][StagedRows<GH>::bytes(GHR)];
  __shared__ __attribute__((aligned(16))) float bias[3 * GH + 32 * GOUT_TILES];
  __shared__ double ys[GNOBS];  // the step's observations

  if constexpr (FILTER) {
    const long f = blockIdx.y;
    a.X = bank_shift(a.X, f * a.bk.x * (long)sizeof(float));
    a.lws = bank_shift(a.lws, f * a.bk.p * (long)sizeof(double));
    a.partials = bank_shift(a.partials, f * (long)gridDim.x * 3 * (long)sizeof(double));
    a.dev = a.dev + f;
    a.batch += (uint32_t)f;
    if (a.par_u_bank != nullptr) a.par_u = a.par_u_bank[f];
  }
  stage_async<G0R, GK0, GP_THREADS>(a.W[0], 0, buf[0]);
#pragma unroll
  for (int l = 0; l < 4; ++l)
    copy_floats(a.b[l], l < 3 ? GH : 32 * GOUT_TILES, bias + l * GH, GP_THREADS);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = lane >> 5;
  const int p = blockIdx.x * GP_TILE + w * 32 + (lane & 31);
  const bool active = p < a.P;
  const int pc = active ? p : 0;

  uint32_t step = a.step;
  const double* y = a.y;
  bool lws_const = false;
  double lws_base = 0.0;
  if constexpr (FILTER) {
    lws_const = a.imp_r != nullptr ? a.imp_r[a.dev->k] != 0
                                   : a.dev->resample != 0 && a.dev->status == BIHIP_OK;
    lws_base = a.dev->logLikelihood;
    step = (uint32_t)(a.dev->k + 1);
    y = a.y_base + (size_t)a.dev->k * a.nobs;
  }

  if (tid < GNOBS) ys[tid] = y[tid];
  __syncthreads();

  // layer-0 operand: inputs 16 c + 8 h + j; the loads without a branch (a
  // particle past the end reads particle 0), so that many are in flight
  uint32_t in0[GK0 / 16][4];
#pragma unroll
  for (int c = 0; c < GK0 / 16; ++c) {
    float u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int f = 16 * c + 8 * h + j;
      float v = 0.0f;
      if (f < GD) {
        v = (a.X[(size_t)f * a.ld + pc] - a.x_shift) * a.x_inv_scale;
      } else if (f < GD + GNOBS) {
        const int o = f - GD;
        v = (float)(ys[o] - (double)a.X[(size_t)(2 * o) * a.ld + pc]) * a.innov_inv;
      } else if (f == GD + GNOBS) {
        v = a.par_u;
      }
      u[j] = v;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) in0[c][j] = pack_bf2(u[2 * j], u[2 * j + 1]);
    // at most 32 loads in flight: all 310 of them would spill
    if ((c & 3) == 3) __builtin_amdgcn_sched_barrier(0);
  }

  uint32_t cur[GH / 16][4], nxt[GH / 16][4];
  // each chunk of rows is copied while the one before is computed
  stage_wait();
  stage_async<G0R, GK0, GP_THREADS>(a.W[0], G0R, buf[1]);
  gelu_tiles<GK0 / 16, GH / 16, GK0, 0, 2>(buf[0], bias, in0, nxt, lane);
  stage_wait();
  stage_async<G0R, GK0, GP_THREADS>(a.W[0], 2 * G0R, buf[0]);
  gelu_tiles<GK0 / 16, GH / 16, GK0, 2, 4>(buf[1], bias, in0, nxt, lane);
  stage_wait();
  stage_async<G0R, GK0, GP_THREADS>(a.W[0], 3 * G0R, buf[1]);
  gelu_tiles<GK0 / 16, GH / 16, GK0, 4, 6>(buf[0], bias, in0, nxt, lane);
  stage_wait();
  stage_async<GHR, GH, GP_THREADS>(a.W[1], 0, buf[0]);
  gelu_tiles<GK0 / 16, GH / 16, GK0, 6, 8>(buf[1], bias, in0, nxt, lane);
  stage_wait();
  stage_async<GHR, GH, GP_THREADS>(a.W[1], GHR, buf[1]);
  gelu_tiles<GH / 16, GH / 16, GH, 0, 4>(buf[0], bias + GH, nxt, cur, lane);
  stage_wait();
  stage_async<GHR, GH, GP_THREADS>(a.W[2], 0, buf[0]);
  gelu_tiles<GH / 16, GH / 16, GH, 4, 8>(buf[1], bias + GH, nxt, cur, lane);
  stage_wait();
  stage_async<GHR, GH, GP_THREADS>(a.W[2], GHR, buf[1]);
  gelu_tiles<GH / 16, GH / 16, GH, 0, 4>(buf[0], bias + 2 * GH, cur, nxt, lane);
  stage_wait();
  stage_async<GHR, GH, GP_THREADS>(a.W[3], 0, buf[0]);
  gelu_tiles<GH / 16, GH / 16, GH, 4, 8>(buf[1], bias + 2 * GH, cur, nxt, lane);

  // output layer in chunks of four tiles; each tile: 16 dimensions (m, s)
  const double inv_obs = 1.0 / a.obs_sd;
  const double c_obs = -HALF_LOG_TWO_PI - log(a.obs_sd);
  double acc_w = 0.0;
  // this lane's states of output tile t (dimensions 16 t + 8 q + 4 h + i), read
  // one tile ahead of their use
  auto load_tile = [&](int t, float (&x)[8]) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (16 * t + 8 * q < GD) x[4 * q + i] = a.X[(size_t)(16 * t + 8 * q + 4 * h + i) * a.ld + pc];
  };
  float xn[8];
  load_tile(0, xn);
  // chunk AT of up to four tiles, in buffer AT % 2
  auto chunk = [&](auto at_c) {
    constexpr int AT = decltype(at_c)::value, T0 = 4 * AT;
    constexpr int NT = GOUT_TILES - T0 < 4 ? GOUT_TILES - T0 : 4;
    constexpr int LEFT = GOUT_TILES - T0 - 4;  // tiles after this chunk
    stage_wait();
    if constexpr (LEFT > 0)
      stage_async<32 * (LEFT < 4 ? LEFT : 4), GH, GP_THREADS>(a.W[3], 32 * (T0 + 4),
                                                              buf[(AT + 1) & 1]);
#pragma unroll
    for (int dt = 0; dt < NT; ++dt) {
      const int t = T0 + dt;
      float xt[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) xt[i] = xn[i];
      if (t + 1 < GOUT_TILES) load_tile(t + 1, xn);
      const f32x16 o =
          linear_tile<GH / 16, GH, true>(buf[AT & 1], dt, t, bias + 3 * GH, nxt, lane);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (16 * t + 8 * q < GD) {
          const int f0 = 16 * t + 8 * q + 4 * h;  // dimensions f0 .. f0 + 3
          float z[4];
          normals4<float>(a.seed, (uint32_t)p, step, TAG_NOISE, a.batch, (uint32_t)(f0 >> 2), z);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int f = f0 + i;
            const float m = o[4 * q + i], s = o[8 + 4 * q + i];
            const float d = m + __expf(0.5f * s) * z[i];  // (x' - Phi) / q
            const float x = xt[4 * q + i] + a.q * d;
            xt[4 * q + i] = x;
            acc_w += (double)(-0.5f * d * d + 0.5f * z[i] * z[i] + 0.5f * s);
            if ((i & 1) == 0) {
              const double e = (ys[f >> 1] - (double)x) * inv_obs;
              acc_w += -0.5 * (e * e) + c_obs;
            }
          }
          if (active) {
#pragma unroll
            for (int i = 0; i < 4; ++i) a.X[(size_t)(f0 + i) * a.ld + p] = xt[4 * q + i];
          }
          // keep the sum here: moved to its use after the last tile, it would
          // hold every tile's values in registers until then
          asm volatile("" : "+v"(acc_w));
        }
      }
    }
  };
  static_assert(GOUT_TILES > 12 && GOUT_TILES <= 16, "four chunks");
  chunk(std::integral_constant<int, 0>{});
  chunk(std::integral_constant<int, 1>{});
  chunk(std::integral_constant<int, 2>{});
  chunk(std::integral_constant<int, 3>{});
  acc_w += __shfl_xor(acc_w, 32, WAVE);  // the particle's other half-wave
  if constexpr (FILTER) {
    double lw = __builtin_nan("");
    if (active && h == 0) {
      lw = (lws_const ? lws_base : a.lws[p]) + acc_w;
      a.lws[p] = lw;
    }
    block_weight_partial<GP_THREADS>(lw, a.partials + 3 * blockIdx.x);
  } else {
    if (active && h == 0) a.inc[p] = acc_w;
  }
}

}  // namespace

int guided_blocks(int P) { return ceil_div(P, GP_TILE); }

int launch_guided(const GuidedLaunch& L, hipStream_t s) {
  const MlpView& n = L.net;
  if (n.L != 4 || n.dims[0] != GD + GNOBS + 1 || n.dims[1] != GH || n.dims[2] != GH ||
      n.dims[3] != GH || n.dims[4] != 2 * GD)
    return set_error(BIHIP_EINVAL, "the guided proposal is built for a 301-256-256-256-400 network");
  if (L.P <= 0) return BIHIP_OK;
  if (L.ld < L.P) return set_error(BIHIP_EINVAL, "ld < P");
  GuidedArgs a{};
  for (int l = 0; l < n.L; ++l) {
    a.W[l] = L.Winf[l];
    a.b[l] = L.binf[l];
  }
  a.x_shift = L.x_shift;
  a.x_inv_scale = 1.0f / L.x_scale;
  a.innov_inv = (float)(1.0 / L.innov_scale);
  a.par_u = (float)((L.par - L.par_shift) / L.par_scale);
  a.X = static_cast<float*>(L.X);
  a.ld = L.ld;
  a.P = L.P;
  a.y = L.y;
  a.seed = L.seed;
  a.batch = L.batch;
  a.step = L.step;
  a.q = L.noise_sd;
  a.obs_sd = L.obs_sd;
  a.dev = L.dev;
  a.y_base = L.y_base;
  a.nobs = L.nobs;
  a.lws = L.lws;
  a.partials = L.partials;
  a.inc = L.inc;
  a.imp_r = L.imp_r;
  a.bk = L.bk;
  a.par_u_bank = L.par_u_bank;
  const int banks = L.banks > 1 ? L.banks : 1;
  if (banks > 1 && L.dev == nullptr)
    return set_error(BIHIP_EINVAL, "a bank runs the guided proposal as a filter step");
  const dim3 grid(guided_blocks(L.P), banks), block(GP_THREADS);
  if (L.dev != nullptr) {
    if (L.lws == nullptr || L.partials == nullptr || L.y_base == nullptr)
      return set_error(BIHIP_EINVAL, "the guided filter step needs the filter's state");
    hipLaunchKernelGGL((k_guided<true>), grid, block, 0, s, a);
  } else {
    if (L.y == nullptr || L.inc == nullptr)
      return set_error(BIHIP_EINVAL, "the guided proposal needs observations and an output");
    hipLaunchKernelGGL((k_guided<false>), grid, block, 0, s, a);
  }
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

}  // namespace bihip
