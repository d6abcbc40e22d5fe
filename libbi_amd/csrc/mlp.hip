// BF16 MFMA kernels of the multilayer perceptron: the tiled GEMM with fused
// epilogues of the forward and backward passes, the loss, weight and bias
// gradients split over the batch, their sums with the Adam step, the inference
// copy of the weights, and input conversion.
//
// The network has no counterpart in the reference (LibBi has no learned
// components): it is the learned surrogate flow and guided proposal built
// beside the bootstrap filter.  Matrices are row-major; bfloat16 operands,
// FP32 accumulation (v_mfma_f32_32x32x16_bf16).
#include "internal.hpp"
#include "mlp.hpp"

namespace bihip {

namespace {

// K steps of 64: the tiles of one step are 2 loads a thread and operand, and a
// 256-wide layer takes four round trips to memory instead of eight (forward
// GEMM of 4096 x 256 x 256 8.4 -> 6.6 us).
constexpr int GB_M = 64, GB_N = 64, GB_K = 64, LDS_K = GB_K + 8;  // +8: bank spread

// Products are computed in 64 x 64 tiles, four waves of 32 x 32.  Operand tiles
// are staged k-contiguous in LDS whatever the global orientation, so every
// fragment read is one 16-byte LDS load.
//
// One 64 x 64 operand tile of K step k0 into LDS, k-contiguous: rows of X from
// r0 (TRANS false: X[(r0 + r) ld + k0 + k], true: X[(k0 + k) ld + r0 + r]).
template <bool TRANS>
struct TileLoad {
  u16x8 v[2];
  __device__ __forceinline__ void load(const uint16_t* X, long ld, int r0, int k0, int tid) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int a = (tid >> 3) + 32 * u, b = (tid & 7) * 8;
      v[u] = TRANS ? *reinterpret_cast<const u16x8*>(X + (size_t)(k0 + a) * ld + r0 + b)
                   : *reinterpret_cast<const u16x8*>(X + (size_t)(r0 + a) * ld + k0 + b);
    }
  }
  __device__ __forceinline__ void store(uint16_t* S, int tid) const {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int a = (tid >> 3) + 32 * u, b = (tid & 7) * 8;
      if (TRANS) {
#pragma unroll
        for (int j = 0; j < 8; ++j) S[(b + j) * LDS_K + a] = v[u][j];
      } else {
        *reinterpret_cast<u16x8*>(&S[a * LDS_K + b]) = v[u];
      }
    }
  }
};

// acc += A B over K steps [kbeg, kend) of a 64 x 64 tile, four waves of 32 x 32;
// the next step's tiles are loaded while this one is computed.  each(As): called
// with every staged A tile.
template <bool TA, bool TB, class Each>
__device__ __forceinline__ void gemm_tile(const uint16_t* A, long lda, const uint16_t* B, long ldb,
                                          int m0, int n0, int kbeg, int kend, uint16_t* As,
                                          uint16_t* Bs, f32x16& acc, Each each) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  TileLoad<TA> ta;
  TileLoad<!TB> tb;
  ta.load(A, lda, m0, kbeg, tid);
  tb.load(B, ldb, n0, kbeg, tid);
  for (int k0 = kbeg; k0 < kend; k0 += GB_K) {
    ta.store(As, tid);
    tb.store(Bs, tid);
    __syncthreads();
    if (k0 + GB_K < kend) {
      ta.load(A, lda, m0, k0 + GB_K, tid);
      tb.load(B, ldb, n0, k0 + GB_K, tid);
    }
    each(As);
#pragma unroll
    for (int kk = 0; kk < GB_K; kk += 16) {
      const u16x8 a = *reinterpret_cast<const u16x8*>(
          &As[(wm * 32 + (lane & 31)) * LDS_K + kk + 8 * (lane >> 5)]);
      const u16x8 b = *reinterpret_cast<const u16x8*>(
          &Bs[(wn * 32 + (lane & 31)) * LDS_K + kk + 8 * (lane >> 5)]);
      acc = mfma32(a, b, acc);
    }
    __syncthreads();
  }
}

// C = A op(B), with B transposed in the forward products.
template <int EPI>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t As[GB_M * LDS_K];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[GB_N * LDS_K];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1;
  const int m0 = blockIdx.x * GB_M, n0 = blockIdx.y * GB_N;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  gemm_tile<false, EPI != EPI_GELU_GRAD>(g.A, g.lda, g.B, g.ldb, m0, n0, 0, g.K, As, Bs, acc,
                                         [](const uint16_t*) {});
  const int col = n0 + wn * 32 + (lane & 31);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = m0 + wm * 32 + acc_row(r, lane);
    const float v = acc[r];
    if constexpr (EPI == EPI_BIAS_GELU) {
      const float z = v + g.bias[col];
      g.Cf[(size_t)row * g.ldc + col] = z;
      g.Cb[(size_t)row * g.ldcb + col] = f2bf(gelu_f(z));
    } else if constexpr (EPI == EPI_BIAS) {
      g.Cf[(size_t)row * g.ldc + col] = v + g.bias[col];
    } else {  // EPI_GELU_GRAD
      g.Cb[(size_t)row * g.ldcb + col] = f2bf(v * gelu_grad_f(g.Zprev[(size_t)row * g.ldz + col]));
    }
  }
}

// Y[i][j] = bf16(X[src(i)][j]) for j < d, 0 for d <= j < ldy, and rows i >= n zero.
__global__ void k_rows_to_bf16(const float* X, long ldx, const long* idx, int n, int rows, int d,
                               uint16_t* Y, int ldy) {
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (long)rows * ldy) return;
  const int i = (int)(g / ldy), j = (int)(g % ldy);
  float v = 0.0f;
  if (i < n && j < d) {
    const long src = idx != nullptr ? idx[i] : i;
    v = X[src * ldx + j];
  }
  Y[g] = f2bf(v);
}

// dY = bf16(2 (Y - T) / (n d)) for the first n rows and d columns (0 elsewhere),
// and per-block partial sums of (Y - T)^2.
__global__ __launch_bounds__(256) void k_mse_grad(const float* Y, int ldy, const float* T, long ldt,
                                                  const long* idx, int n, int rows, int d,
                                                  float scale, uint16_t* dY, float* partial) {
  __shared__ float red[256];
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  float sq = 0.0f;
  if (g < (long)rows * ldy) {
    const int i = (int)(g / ldy), j = (int)(g % ldy);
    float gr = 0.0f;
    if (i < n && j < d) {
      const long src = idx != nullptr ? idx[i] : i;
      const float e = Y[(size_t)i * ldy + j] - T[src * ldt + j];
      sq = e * e;
      gr = scale * e;
    }
    dY[g] = f2bf(gr);
  }
  red[threadIdx.x] = sq;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// Gaussian negative log-likelihood: Y holds the mean (columns < m) and the log
// variance (columns m .. 2m - 1) for m targets.  dY = bf16 of the gradient of
// sum [(t - mu)^2 e^{-s} + s] / (2 n m); partial sums of the per-target terms.
__global__ __launch_bounds__(256) void k_gauss_grad(const float* Y, int ldy, const float* T,
                                                    long ldt, const long* idx, int n, int rows,
                                                    int m, float scale, uint16_t* dY,
                                                    float* partial) {
  __shared__ float red[256];
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  float term = 0.0f;
  if (g < (long)rows * ldy) {
    const int i = (int)(g / ldy), j = (int)(g % ldy);
    float gr = 0.0f;
    if (i < n && j < 2 * m) {
      const int o = j < m ? j : j - m;
      const long src = idx != nullptr ? idx[i] : i;
      const float mu = Y[(size_t)i * ldy + o], lv = Y[(size_t)i * ldy + m + o];
      const float e = T[src * ldt + o] - mu, iv = __expf(-lv), q = e * e * iv;
      if (j < m) {
        gr = -scale * e * iv;
        term = 0.5f * (q + lv);
      } else {
        gr = 0.5f * scale * (1.0f - q);
      }
    }
    dY[g] = f2bf(gr);
  }
  red[threadIdx.x] = term;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// Weight and bias gradients of several layers in one launch, split over the
// batch: block b takes a 64 x 64 tile of dZ^T A of one layer over one split of
// the rows and stores its partial sums; the blocks of a layer's first tile
// column also sum the columns of dZ (the bias gradient) from the tiles they
// stage, thread (m, eight row slots) adding rows slot, slot + 32, ... in order
// and then the 32 slots in order.  A layer alone is at most 256 blocks of four
// K steps: 9.3 us each, and 4.2 + 3.4 us for its column sums in launches of
// their own; together 17.5 us for four layers.
__global__ __launch_bounds__(256) void k_weight_grads(WeightGradArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t As[GB_M * LDS_K];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[GB_N * LDS_K];
  __shared__ float red[32][64 + 1];
  int l = 0;
  while (l + 1 < g.n && (int)blockIdx.x >= g.layer[l + 1].block0) ++l;
  const WeightGradLayer& y = g.layer[l];
  const int nt = y.N / GB_N, mt = y.M / GB_M;
  int b = (int)blockIdx.x - y.block0;
  const int n0 = b % nt * GB_N;
  b /= nt;
  const int m0 = b % mt * GB_M, z = b / mt;
  const int kbeg = z * g.ksplit, kend = min(kbeg + g.ksplit, g.rows);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  float col[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) col[j] = 0.0f;
  const bool sums = n0 == 0;
  const int m = tid & 63, slot = (tid >> 6) * 8;
  gemm_tile<true, false>(y.dZ, y.ldz, y.act, y.lda, m0, n0, kbeg, kend, As, Bs, acc,
                         [&](const uint16_t* S) {
                           if (!sums) return;
                           const u16x8 a =
                               *reinterpret_cast<const u16x8*>(&S[m * LDS_K + slot]);
                           const u16x8 c =
                               *reinterpret_cast<const u16x8*>(&S[m * LDS_K + slot + 32]);
#pragma unroll
                           for (int j = 0; j < 8; ++j) col[j] += bf2f(a[j]);
#pragma unroll
                           for (int j = 0; j < 8; ++j) col[j] += bf2f(c[j]);
                         });
  float* part = y.partW + (size_t)z * y.M * y.N;
  const int c0 = n0 + (w & 1) * 32 + (lane & 31);
#pragma unroll
  for (int r = 0; r < 16; ++r)
    part[(size_t)(m0 + (w >> 1) * 32 + acc_row(r, lane)) * y.N + c0] = acc[r];
  if (!sums) return;
#pragma unroll
  for (int j = 0; j < 8; ++j) red[slot + j][m] = col[j];
  __syncthreads();
  if (tid < 64) {
    float t = 0.0f;
    for (int q = 0; q < 32; ++q) t += red[q][tid];
    y.partb[(size_t)z * y.M + m0 + tid] = t;
  }
}

// The splits of several parameter segments summed in the order s = 0, 1, ...,
// S-1 (four parameters a thread, eight splits in flight), and what becomes of
// the sums: the gradient (adam == 0), or an Adam step (Kingma & Ba 2015, with
// bias correction) on the FP32 parameters with their bfloat16 copy.  One more
// block (loss_out) sums the minibatch's loss terms.  One launch for all layers;
// as a sum per weight and bias array, two Adam launches and one for the loss it
// was eleven of 2.4 to 3.5 us.
__global__ __launch_bounds__(256) void k_update(UpdateArgs a) {
  if (a.loss_out != nullptr && blockIdx.x == gridDim.x - 1) {
    __shared__ float red[256];
    float s = 0.0f;
    for (int i = threadIdx.x; i < a.nloss; i += 256) s += a.loss[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
      __syncthreads();
    }
    if (threadIdx.x == 0) *a.loss_out = red[0];
    return;
  }
  int q = 0;
  while (q + 1 < a.n && (int)blockIdx.x >= a.seg[q + 1].block0) ++q;
  const UpdateSegment& e = a.seg[q];
  const long i = ((long)((int)blockIdx.x - e.block0) * 256 + threadIdx.x) * 4;
  if (i >= e.count) return;
  float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
  int z = 0;
  for (; z + 8 <= a.S; z += 8) {
    float4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      v[u] = *reinterpret_cast<const float4*>(e.part + (size_t)(z + u) * e.count + i);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      g.x += v[u].x;
      g.y += v[u].y;
      g.z += v[u].z;
      g.w += v[u].w;
    }
  }
  for (; z < a.S; ++z) {
    const float4 v = *reinterpret_cast<const float4*>(e.part + (size_t)z * e.count + i);
    g.x += v.x;
    g.y += v.y;
    g.z += v.z;
    g.w += v.w;
  }
  const long k = e.off + i;
  if (a.adam == 0) {
    *reinterpret_cast<float4*>(a.G + k) = g;
    return;
  }
  float gr[4] = {g.x, g.y, g.z, g.w};
  float4 m1 = *reinterpret_cast<float4*>(a.M1 + k), m2 = *reinterpret_cast<float4*>(a.M2 + k),
         w = *reinterpret_cast<float4*>(a.P + k);
  float* m1v = &m1.x;
  float* m2v = &m2.x;
  float* wv = &w.x;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    // which of the two products is fused is stated: a training's parameters
    // follow from it
    const float x = __builtin_fmaf(1.0f - a.b1, gr[u], a.b1 * m1v[u]);
    const float y = __builtin_fmaf((1.0f - a.b2) * gr[u], gr[u], a.b2 * m2v[u]);
    m1v[u] = x;
    m2v[u] = y;
    wv[u] = wv[u] - a.lr * (x / a.bc1) / (sqrtf(y / a.bc2) + a.eps);
  }
  *reinterpret_cast<float4*>(a.M1 + k) = m1;
  *reinterpret_cast<float4*>(a.M2 + k) = m2;
  *reinterpret_cast<float4*>(a.P + k) = w;
  if (k < a.nW) {
    uint2 h;
    h.x = pack_bf2(w.x, w.y);
    h.y = pack_bf2(w.z, w.w);
    *reinterpret_cast<uint2*>(a.Wbf + k) = h;
  }
}

__global__ void k_to_bf16(const float* x, long n, uint16_t* y) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

// Source row of row n of the inference weights' layer l: natural, or for an
// interleaved output layer (blocks of 2 interleave rows: m of outputs
// t interleave .., then s of the same ones) the row of that number; -1: a row
// of zeros.
__device__ __forceinline__ int inference_row(const InferenceWeightsArgs& a, int l, int n) {
  if (l != a.L - 1 || a.interleave <= 0) return n;
  const int oi = a.interleave, t = n / (2 * oi), r = n % (2 * oi);
  const int dim = t * oi + (r < oi ? r : r - oi);
  return dim < a.dout / 2 ? (r < oi ? dim : a.dout / 2 + dim) : -1;
}

// The inference copy of the weights and biases: bfloat16 weights, the input
// columns of layers l >= 1 in the order the accumulators of the layer before
// leave them (position 16 c + q holds input 16 c + 8 ((q % 8) / 4) + 4 (q / 8)
// + q % 4).  A thread writes eight consecutive weights, two runs of four
// inputs, or one bias (the padded widths are multiples of 64).  Bound by its
// launch (297 k weights: 3.5 us); laid out on the host behind a copy in each
// direction it took 0.4 ms of every call that uses a network.
__global__ __launch_bounds__(256) void k_inference_weights(InferenceWeightsArgs a) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  const long nw8 = a.nW / 8;
  if (g < nw8) {
    int l = 0;
    while (l + 1 < a.L && a.offW[l + 1] <= 8 * g) ++l;
    const int K = a.pad[l];
    const long e = 8 * g - a.offW[l];
    const int n = (int)(e / K), k = (int)(e % K);
    const int row = inference_row(a, l, n);
    float4 v0 = make_float4(0.f, 0.f, 0.f, 0.f), v1 = v0;
    if (row >= 0) {
      const float* src = a.P + a.offW[l] + (long)row * K;
      const int k0 = l == 0 ? k : (k & ~15) + ((k & 8) >> 1);
      v0 = *reinterpret_cast<const float4*>(src + k0);
      v1 = *reinterpret_cast<const float4*>(src + k0 + (l == 0 ? 4 : 8));
    }
    *reinterpret_cast<u32v4*>(a.W + 8 * g) =
        u32v4{pack_bf2(v0.x, v0.y), pack_bf2(v0.z, v0.w), pack_bf2(v1.x, v1.y),
              pack_bf2(v1.z, v1.w)};
  } else if (g - nw8 < a.nb) {
    const long i = g - nw8;
    int l = 0;
    while (l + 1 < a.L && a.offb[l + 1] <= i) ++l;
    const int row = inference_row(a, l, (int)(i - a.offb[l]));
    a.b[i] = row >= 0 ? a.P[a.nW + a.offb[l] + row] : 0.0f;
  }
}

}  // namespace

int launch_gemm(const GemmArgs& g, int epi, hipStream_t s) {
  // the kernel's tiling assumptions, checked here so that no access leaves the operands
  if (g.M <= 0 || g.N <= 0 || g.K <= 0 || g.M % GB_M || g.N % GB_N || g.K % GB_K ||
      g.lda % 8 || g.ldb % 8)
    return set_error(BIHIP_EINVAL, "GEMM shape %dx%dx%d (lda %ld, ldb %ld) off the 64x64x64 "
                     "tiling", g.M, g.N, g.K, g.lda, g.ldb);
  if (((uintptr_t)g.A | (uintptr_t)g.B) & 15)
    return set_error(BIHIP_EINVAL, "GEMM operands must be 16-byte aligned");
  const dim3 grid(g.M / GB_M, g.N / GB_N), block(256);
  switch (epi) {
    case EPI_BIAS_GELU: hipLaunchKernelGGL(k_gemm<EPI_BIAS_GELU>, grid, block, 0, s, g); break;
    case EPI_BIAS: hipLaunchKernelGGL(k_gemm<EPI_BIAS>, grid, block, 0, s, g); break;
    case EPI_GELU_GRAD: hipLaunchKernelGGL(k_gemm<EPI_GELU_GRAD>, grid, block, 0, s, g); break;
    default: return set_error(BIHIP_EINVAL, "unknown GEMM epilogue %d", epi);
  }
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_rows_to_bf16(const float* X, long ldx, const long* idx, int n, int rows, int d,
                        uint16_t* Y, int ldy, hipStream_t s) {
  const long tot = (long)rows * ldy;
  if (tot <= 0) return BIHIP_OK;
  hipLaunchKernelGGL(k_rows_to_bf16, dim3(ceil_div(tot, 256)), dim3(256), 0, s, X, ldx, idx, n,
                     rows, d, Y, ldy);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_mse_grad(const float* Y, int ldy, const float* T, long ldt, const long* idx, int n,
                    int rows, int d, float scale, uint16_t* dY, float* partial, int* nblocks,
                    hipStream_t s) {
  const long tot = (long)rows * ldy;
  *nblocks = ceil_div(tot, 256);
  hipLaunchKernelGGL(k_mse_grad, dim3(*nblocks), dim3(256), 0, s, Y, ldy, T, ldt, idx, n, rows, d,
                     scale, dY, partial);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_gauss_grad(const float* Y, int ldy, const float* T, long ldt, const long* idx, int n,
                      int rows, int m, float scale, uint16_t* dY, float* partial, int* nblocks,
                      hipStream_t s) {
  const long tot = (long)rows * ldy;
  *nblocks = ceil_div(tot, 256);
  hipLaunchKernelGGL(k_gauss_grad, dim3(*nblocks), dim3(256), 0, s, Y, ldy, T, ldt, idx, n, rows,
                     m, scale, dY, partial);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_weight_grads(const WeightGradArgs& g, hipStream_t s) {
  if (g.n <= 0) return BIHIP_OK;
  if (g.rows <= 0 || g.rows % GB_K || g.ksplit <= 0 || g.ksplit % GB_K)
    return set_error(BIHIP_EINVAL, "weight gradients of %d rows (split %d) off the 64-row steps",
                     g.rows, g.ksplit);
  const int S = ceil_div(g.rows, g.ksplit);
  long blocks = 0;
  for (int l = 0; l < g.n; ++l) {
    const WeightGradLayer& y = g.layer[l];
    if (y.M <= 0 || y.N <= 0 || y.M % GB_M || y.N % GB_N || y.ldz % 8 || y.lda % 8 ||
        (((uintptr_t)y.dZ | (uintptr_t)y.act) & 15) || y.block0 != blocks)
      return set_error(BIHIP_EINVAL, "weight gradient %dx%d off the 64x64 tiling", y.M, y.N);
    blocks += (long)(y.M / GB_M) * (y.N / GB_N) * S;
  }
  hipLaunchKernelGGL(k_weight_grads, dim3(blocks), dim3(256), 0, s, g);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_update(const UpdateArgs& a, hipStream_t s) {
  long blocks = 0;
  for (int q = 0; q < a.n; ++q) {
    const UpdateSegment& e = a.seg[q];
    if (e.count % 4 || e.off % 4 || e.block0 != blocks || ((uintptr_t)e.part & 15))
      return set_error(BIHIP_EINVAL, "parameter segments of padded widths are needed");
    blocks += ceil_div(e.count / 4, 256);
  }
  if (a.loss_out != nullptr) ++blocks;
  if (blocks == 0) return BIHIP_OK;
  hipLaunchKernelGGL(k_update, dim3(blocks), dim3(256), 0, s, a);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_inference_weights(const InferenceWeightsArgs& a, hipStream_t s) {
  // vector accesses: widths of a multiple of 64 from aligned arenas
  for (int l = 0; l < a.L; ++l)
    if (a.pad[l] % 16 || a.offW[l] % 8)
      return set_error(BIHIP_EINVAL, "inference weights need padded widths");
  hipLaunchKernelGGL(k_inference_weights, dim3(ceil_div(a.nW / 8 + a.nb, 256)), dim3(256), 0, s,
                     a);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_to_bf16(const float* x, long n, uint16_t* y, hipStream_t s) {
  if (n <= 0) return BIHIP_OK;
  hipLaunchKernelGGL(k_to_bf16, dim3(ceil_div(n, 256)), dim3(256), 0, s, x, n, y);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

}  // namespace bihip
