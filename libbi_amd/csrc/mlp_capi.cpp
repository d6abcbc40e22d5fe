// C ABI of the BF16 MFMA multilayer perceptron (bihip_mlp_*, declared in include/bihip.h).
//
// Layers l = 0..L-1 map d_l -> d_{l+1}: z = W_l a + b_l, GELU z sigma(1.702 z)
// on hidden layers, linear output.  Every width is padded to a multiple of 64 on the
// device (padded weights, inputs and output errors are zero, so the padding
// never reaches a result).  Parameters are kept in FP32 (the Adam master
// copy) and, for the weights, in bfloat16 for the matrix cores.  The flat host
// layout is, per layer, W_l row-major [d_{l+1}][d_l] then b_l.
#include <cmath>
#include <cstring>
#include <numeric>
#include <mutex>
#include <utility>
#include <vector>

#include "internal.hpp"

using namespace bihip;

namespace {
constexpr uint32_t TAG_MLP_INIT = 11;
constexpr uint32_t TAG_MLP_BATCH = 12;
constexpr long UNIF_CHUNK = 1L << 22;  // uniforms of the shuffle held at once
int pad64(int d) { return (d + 63) / 64 * 64; }
}  // namespace

struct bihip_mlp {
  bihip_ctx* ctx = nullptr;
  int L = 0;
  std::vector<int> dims, pad;
  std::vector<long> offW, offb;  // offsets in the FP32 arenas: [all W | all b]
  long nW = 0, ntot = 0;
  float *P = nullptr, *G = nullptr, *M1 = nullptr, *M2 = nullptr;
  uint16_t* Wbf = nullptr;       // bf16 weights, same offsets as the W part
  long adam_t = 0;
  int loss = BIHIP_LOSS_MSE;
  // workspace for batches of up to cap rows
  int cap = 0;
  uint16_t* X0 = nullptr;
  std::vector<float*> Z;         // pre-activations / output, per layer
  std::vector<uint16_t*> A;      // bf16 activations, A[l] = input of layer l (l >= 1)
  std::vector<uint16_t*> dZ;     // bf16 errors per layer output
  float* part = nullptr;         // split-K partials
  long part_n = 0;
  float* lossp = nullptr;
  uint16_t* Winf = nullptr;      // inference copy of the weights (permuted columns)
  float* binf = nullptr;         // inference copy of the biases (row order of Winf)
  // reads of Winf and binf queued on other streams than the network's: the next
  // layout waits for them
  std::mutex readers_lock;
  std::vector<std::pair<hipStream_t, hipEvent_t>> readers;
};

namespace {

void free_work(bihip_mlp* m) {
  dfree(m->X0);
  for (auto p : m->Z) dfree(p);
  for (auto p : m->A) dfree(p);
  for (auto p : m->dZ) dfree(p);
  dfree(m->part);
  dfree(m->lossp);
  m->X0 = nullptr;
  m->Z.clear();
  m->A.clear();
  m->dZ.clear();
  m->part = m->lossp = nullptr;
  m->cap = 0;
}

constexpr int KSPLIT = 256;  // batch rows per split of the weight-gradient GEMMs
// Floats of partial sums up to which all layers' gradients share one launch
// (larger networks take a layer at a time).
constexpr long PART_GROUP = 1L << 26;

int ensure_work(bihip_mlp* m, int rows) {
  if (rows <= m->cap) return BIHIP_OK;
  free_work(m);
  const int L = m->L;
  int rc;
  if ((rc = dalloc(&m->X0, (size_t)rows * m->pad[0]))) return rc;
  m->Z.assign(L, nullptr);
  m->A.assign(L, nullptr);
  m->dZ.assign(L, nullptr);
  long maxw = 0;
  for (int l = 0; l < L; ++l) {
    if ((rc = dalloc(&m->Z[l], (size_t)rows * m->pad[l + 1]))) return rc;
    if ((rc = dalloc(&m->dZ[l], (size_t)rows * m->pad[l + 1]))) return rc;
    if (l + 1 < L && (rc = dalloc(&m->A[l + 1], (size_t)rows * m->pad[l + 1]))) return rc;
    maxw = std::max(maxw, (long)m->pad[l + 1] * (m->pad[l] + 1));
  }
  const int S = (rows + KSPLIT - 1) / KSPLIT;
  // one layer's partial sums, or all of them where they stay small
  m->part_n = std::max(maxw * S, std::min(m->ntot * S, PART_GROUP));
  if ((rc = dalloc(&m->part, (size_t)m->part_n))) return rc;
  if ((rc = dalloc(&m->lossp, (size_t)rows * m->pad[L] / 256 + 1))) return rc;
  m->cap = rows;
  return BIHIP_OK;
}

// forward over rows (multiple of 64) already in X0
int forward(bihip_mlp* m, int rows, hipStream_t s) {
  const int L = m->L;
  for (int l = 0; l < L; ++l) {
    GemmArgs g{};
    g.A = l == 0 ? m->X0 : m->A[l];
    g.lda = m->pad[l];
    g.B = m->Wbf + m->offW[l];
    g.ldb = m->pad[l];
    g.M = rows;
    g.N = m->pad[l + 1];
    g.K = m->pad[l];
    g.bias = m->P + m->offb[l];
    g.Cf = m->Z[l];
    g.ldc = m->pad[l + 1];
    g.Cb = l + 1 < L ? m->A[l + 1] : nullptr;
    g.ldcb = m->pad[l + 1];
    int rc = launch_gemm(g, l + 1 < L ? EPI_BIAS_GELU : EPI_BIAS, s);
    if (rc) return rc;
  }
  return BIHIP_OK;
}

// Backward from dZ[L-1] (already set): the errors of the layers, then their
// gradients in as few launches as the partial sums' workspace allows (usually
// one), each followed by the launch that sums them into the gradient arena G or
// takes the Adam step `u` describes.
int backward(bihip_mlp* m, int rows, const UpdateArgs& u, hipStream_t s) {
  int rc;
  for (int l = m->L - 1; l > 0; --l) {
    GemmArgs h{};  // dZ_{l-1} = (dZ_l W_l) * GELU'(Z_{l-1})
    h.A = m->dZ[l];
    h.lda = m->pad[l + 1];
    h.B = m->Wbf + m->offW[l];
    h.ldb = m->pad[l];
    h.M = rows;
    h.N = m->pad[l];
    h.K = m->pad[l + 1];
    h.Zprev = m->Z[l - 1];
    h.ldz = m->pad[l];
    h.Cb = m->dZ[l - 1];
    h.ldcb = m->pad[l];
    if ((rc = launch_gemm(h, EPI_GELU_GRAD, s))) return rc;
  }
  const int ksplit = std::min(rows, KSPLIT), S = (rows + ksplit - 1) / ksplit;
  for (int l = 0; l < m->L;) {
    WeightGradArgs g{};  // dW_l = dZ_l^T A_l, split over the batch
    g.rows = rows;
    g.ksplit = ksplit;
    UpdateArgs a = u;
    a.S = S;
    a.P = m->P;
    a.G = m->G;
    a.M1 = m->M1;
    a.M2 = m->M2;
    a.Wbf = m->Wbf;
    a.nW = m->nW;
    long used = 0, gblocks = 0, ublocks = 0;
    for (; l < m->L; ++l) {
      const int M = m->pad[l + 1], N = m->pad[l];
      const long cw = (long)M * N, need = (cw + M) * S;
      if (g.n > 0 && used + need > m->part_n) break;
      WeightGradLayer& y = g.layer[g.n++];
      y.dZ = m->dZ[l];
      y.ldz = M;
      y.act = l == 0 ? m->X0 : m->A[l];
      y.lda = N;
      y.M = M;
      y.N = N;
      y.block0 = (int)gblocks;
      y.partW = m->part + used;
      y.partb = y.partW + cw * S;
      gblocks += cw / 4096 * S;
      used += need;
      a.seg[a.n++] = UpdateSegment{y.partW, cw, m->offW[l], (int)ublocks};
      ublocks += (cw / 4 + 255) / 256;
      a.seg[a.n++] = UpdateSegment{y.partb, M, m->offb[l], (int)ublocks};
      ublocks += (M / 4 + 255) / 256;
    }
    if (l < m->L) a.loss_out = nullptr;  // the last launch sums the loss
    if ((rc = launch_weight_grads(g, s)) || (rc = launch_update(a, s))) return rc;
  }
  return BIHIP_OK;
}

// output error dL/dy of the configured loss for n valid rows (rows padded);
// per-block partial sums of the loss terms into m->lossp
int output_error(bihip_mlp* m, const float* T, long ldt, const long* idx, int n, int rows,
                 int* nblocks, hipStream_t s) {
  const int L = m->L, d = m->dims[L];
  if (m->loss == BIHIP_LOSS_GAUSS)
    return launch_gauss_grad(m->Z[L - 1], m->pad[L], T, ldt, idx, n, rows, d / 2,
                             1.0f / ((float)n * (float)(d / 2)), m->dZ[L - 1], m->lossp, nblocks,
                             s);
  return launch_mse_grad(m->Z[L - 1], m->pad[L], T, ldt, idx, n, rows, d,
                         2.0f / ((float)n * (float)d), m->dZ[L - 1], m->lossp, nblocks, s);
}

int targets_per_sample(const bihip_mlp* m) {
  return m->loss == BIHIP_LOSS_GAUSS ? m->dims[m->L] / 2 : m->dims[m->L];
}

// loss and output error; *sumsq gets the summed loss terms
int loss_and_error(bihip_mlp* m, const float* T, long ldt, const long* idx, int n, int rows,
                   double* sumsq, hipStream_t s) {
  int nb = 0;
  int rc = output_error(m, T, ldt, idx, n, rows, &nb, s);
  if (rc) return rc;
  if (sumsq) {
    std::vector<float> h(nb);
    BIHIP_HIP(hipMemcpyAsync(h.data(), m->lossp, sizeof(float) * nb, hipMemcpyDeviceToHost, s));
    BIHIP_HIP(hipStreamSynchronize(s));
    double t = 0.0;
    for (float v : h) t += v;
    *sumsq = t;
  }
  return BIHIP_OK;
}

int upload_params(bihip_mlp* m, const float* flat, hipStream_t s) {
  std::vector<float> P(m->ntot, 0.0f);
  long o = 0;
  for (int l = 0; l < m->L; ++l) {
    const int din = m->dims[l], dout = m->dims[l + 1];
    for (int r = 0; r < dout; ++r)
      for (int c = 0; c < din; ++c) P[m->offW[l] + (long)r * m->pad[l] + c] = flat[o++];
    for (int r = 0; r < dout; ++r) P[m->offb[l] + r] = flat[o++];
  }
  BIHIP_HIP(hipMemcpyAsync(m->P, P.data(), sizeof(float) * m->ntot, hipMemcpyHostToDevice, s));
  int rc = launch_to_bf16(m->P, m->nW, m->Wbf, s);
  if (rc) return rc;
  BIHIP_HIP(hipStreamSynchronize(s));
  return BIHIP_OK;
}

void unpack(const bihip_mlp* m, const std::vector<float>& P, float* flat) {
  long o = 0;
  for (int l = 0; l < m->L; ++l) {
    const int din = m->dims[l], dout = m->dims[l + 1];
    for (int r = 0; r < dout; ++r)
      for (int c = 0; c < din; ++c) flat[o++] = P[m->offW[l] + (long)r * m->pad[l] + c];
    for (int r = 0; r < dout; ++r) flat[o++] = P[m->offb[l] + r];
  }
}

}  // namespace

// Notes that what is queued on `user` so far may read the inference copy.  (A
// captured stream has nothing queued, and an event recorded there would not be
// one of this run.)
static int note_reader(bihip_mlp* m, hipStream_t user) {
  if (user == ctx_stream_of(m->ctx)) return BIHIP_OK;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  BIHIP_HIP(hipStreamIsCapturing(user, &cap));
  if (cap != hipStreamCaptureStatusNone) return BIHIP_OK;
  std::lock_guard<std::mutex> hold(m->readers_lock);
  for (auto& r : m->readers)
    if (r.first == user) {
      BIHIP_HIP(hipEventRecord(r.second, user));
      return BIHIP_OK;
    }
  hipEvent_t e;
  BIHIP_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (hipEventRecord(e, user) != hipSuccess) {
    (void)hipEventDestroy(e);
    return set_error(BIHIP_EHIP, "noting a reader of the network failed");
  }
  m->readers.emplace_back(user, e);
  return BIHIP_OK;
}

// The network's stream waits for the noted reads.
static int await_readers(bihip_mlp* m, hipStream_t s) {
  std::lock_guard<std::mutex> hold(m->readers_lock);
  hipError_t err = hipSuccess;
  for (auto& r : m->readers) {
    const hipError_t e = hipStreamWaitEvent(s, r.second, 0);
    if (err == hipSuccess) err = e;
    (void)hipEventDestroy(r.second);  // takes effect once the event has completed
  }
  m->readers.clear();
  return err == hipSuccess ? BIHIP_OK
                           : set_error(BIHIP_EHIP, "waiting for readers of the network: %s",
                                       hipGetErrorString(err));
}

namespace bihip {
int mlp_inference_weights(bihip_mlp* m, hipStream_t user, const uint16_t* W[MLP_MAX_LAYERS],
                          const float* b[MLP_MAX_LAYERS], int out_interleave) {
  if (m->L > MLP_MAX_LAYERS) return set_error(BIHIP_EINVAL, "too many layers");
  const int L = m->L, dout = m->dims[L];
  if (out_interleave > 0 && (dout % 2 || 2 * ((dout / 2 + out_interleave - 1) / out_interleave) *
                                               out_interleave > m->pad[L]))
    return set_error(BIHIP_EINVAL, "output interleave does not fit the padded width");
  int rc;
  hipStream_t s = ctx_stream_of(m->ctx);
  // a replay would not lay out the weights that the network has by then
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  BIHIP_HIP(hipStreamIsCapturing(s, &cap));
  if (cap != hipStreamCaptureStatusNone)
    return set_error(BIHIP_EHIP, "inference weights are not laid out under stream capture");
  if (m->Winf == nullptr && (rc = dalloc(&m->Winf, m->nW))) return rc;
  if (m->binf == nullptr && (rc = dalloc(&m->binf, m->ntot - m->nW))) return rc;
  InferenceWeightsArgs a{};
  a.P = m->P;
  a.W = m->Winf;
  a.b = m->binf;
  a.L = L;
  a.nW = m->nW;
  a.nb = m->ntot - m->nW;
  a.interleave = out_interleave;
  a.dout = dout;
  for (int l = 0; l <= L; ++l) a.pad[l] = m->pad[l];
  for (int l = 0; l < L; ++l) {
    a.offW[l] = m->offW[l];
    a.offb[l] = m->offb[l] - m->nW;
    W[l] = m->Winf + m->offW[l];
    if (b != nullptr) b[l] = m->binf + a.offb[l];
  }
  if ((rc = note_reader(m, user)) || (rc = await_readers(m, s)) ||
      (rc = launch_inference_weights(a, s)))
    return rc;
  if (user != s) BIHIP_HIP(hipStreamSynchronize(s));  // no order between the streams
  return BIHIP_OK;
}

// Shape of an MLP for the fused inference kernels (surrogate.hip, guided.hip).
MlpView mlp_view(const bihip_mlp* m) {
  MlpView v{};
  v.L = m->L;
  for (int l = 0; l <= m->L && l < MLP_MAX_LAYERS + 1; ++l) {
    v.dims[l] = m->dims[l];
    v.pad[l] = m->pad[l];
  }
  return v;
}
}  // namespace bihip

extern "C" {

int bihip_mlp_create(bihip_ctx* ctx, int nlayers, const int* dims, uint64_t seed,
                     bihip_mlp** out) {
  int rc = ctx_enter_device(ctx);
  if (rc) return rc;
  if (dims == nullptr || out == nullptr) return set_error(BIHIP_EINVAL, "NULL argument");
  if (nlayers < 1 || nlayers > MLP_MAX_LAYERS)
    return set_error(BIHIP_EINVAL, "nlayers must lie in [1, %d]", MLP_MAX_LAYERS);
  for (int l = 0; l <= nlayers; ++l)
    if (dims[l] < 1 || dims[l] > 4096) return set_error(BIHIP_EINVAL, "width %d outside [1,4096]", dims[l]);
  bihip_mlp* m = new bihip_mlp();
  m->ctx = ctx;
  m->L = nlayers;
  m->dims.assign(dims, dims + nlayers + 1);
  for (int l = 0; l <= nlayers; ++l) m->pad.push_back(pad64(dims[l]));
  long o = 0;
  for (int l = 0; l < nlayers; ++l) {
    m->offW.push_back(o);
    o += (long)m->pad[l + 1] * m->pad[l];
  }
  m->nW = o;
  for (int l = 0; l < nlayers; ++l) {
    m->offb.push_back(o);
    o += m->pad[l + 1];
  }
  m->ntot = o;
  if ((rc = dalloc(&m->P, m->ntot)) || (rc = dalloc(&m->G, m->ntot)) ||
      (rc = dalloc(&m->M1, m->ntot)) || (rc = dalloc(&m->M2, m->ntot)) ||
      (rc = dalloc(&m->Wbf, m->nW))) {
    bihip_mlp_destroy(m);
    return rc;
  }
  hipStream_t s = ctx_stream_of(ctx);
  BIHIP_HIP(hipMemsetAsync(m->G, 0, sizeof(float) * m->ntot, s));
  BIHIP_HIP(hipMemsetAsync(m->M1, 0, sizeof(float) * m->ntot, s));
  BIHIP_HIP(hipMemsetAsync(m->M2, 0, sizeof(float) * m->ntot, s));
  // U(-1/sqrt(d_in), 1/sqrt(d_in)) for weights and biases, keyed Philox draws
  std::vector<float> flat((size_t)bihip_mlp_nparams(m));
  long k = 0;
  for (int l = 0; l < nlayers; ++l) {
    const double bound = 1.0 / std::sqrt((double)dims[l]);
    const long cnt = (long)dims[l + 1] * dims[l] + dims[l + 1];
    for (long i = 0; i < cnt; ++i) {
      const double u = bihip_uniform_host(seed, (uint32_t)i, (uint32_t)l, TAG_MLP_INIT, 0);
      flat[k++] = (float)(bound * (2.0 * u - 1.0));
    }
  }
  if ((rc = upload_params(m, flat.data(), s))) {
    bihip_mlp_destroy(m);
    return rc;
  }
  *out = m;
  return BIHIP_OK;
}

int bihip_mlp_destroy(bihip_mlp* m) {
  if (m == nullptr) return BIHIP_OK;
  (void)ctx_enter_device(m->ctx);
  (void)hipStreamSynchronize(ctx_stream_of(m->ctx));
  for (auto& r : m->readers) (void)hipEventDestroy(r.second);
  free_work(m);
  dfree(m->P);
  dfree(m->G);
  dfree(m->M1);
  dfree(m->M2);
  dfree(m->Wbf);
  dfree(m->Winf);
  dfree(m->binf);
  delete m;
  return BIHIP_OK;
}

long bihip_mlp_nparams(const bihip_mlp* m) {
  if (m == nullptr) return -1;
  long n = 0;
  for (int l = 0; l < m->L; ++l) n += (long)m->dims[l + 1] * m->dims[l] + m->dims[l + 1];
  return n;
}

int bihip_mlp_set_params(bihip_mlp* m, const float* flat_host) {
  if (m == nullptr || flat_host == nullptr) return set_error(BIHIP_EINVAL, "NULL argument");
  int rc = ctx_enter_device(m->ctx);
  if (rc) return rc;
  hipStream_t s = ctx_stream_of(m->ctx);
  if ((rc = upload_params(m, flat_host, s))) return rc;
  BIHIP_HIP(hipMemsetAsync(m->M1, 0, sizeof(float) * m->ntot, s));
  BIHIP_HIP(hipMemsetAsync(m->M2, 0, sizeof(float) * m->ntot, s));
  BIHIP_HIP(hipStreamSynchronize(s));
  m->adam_t = 0;
  return BIHIP_OK;
}

int bihip_mlp_get_params(bihip_mlp* m, float* flat_host) {
  if (m == nullptr || flat_host == nullptr) return set_error(BIHIP_EINVAL, "NULL argument");
  int rc = ctx_enter_device(m->ctx);
  if (rc) return rc;
  hipStream_t s = ctx_stream_of(m->ctx);
  std::vector<float> P(m->ntot);
  BIHIP_HIP(hipMemcpyAsync(P.data(), m->P, sizeof(float) * m->ntot, hipMemcpyDeviceToHost, s));
  BIHIP_HIP(hipStreamSynchronize(s));
  unpack(m, P, flat_host);
  return BIHIP_OK;
}

int bihip_mlp_forward(bihip_mlp* m, const float* X_dev, long ldx, long n, float* Y_dev,
                      long ldy) {
  if (m == nullptr || X_dev == nullptr || Y_dev == nullptr)
    return set_error(BIHIP_EINVAL, "NULL argument");
  if (n < 0 || ldx < m->dims[0] || ldy < m->dims[m->L])
    return set_error(BIHIP_EINVAL, "bad n or leading dimensions");
  int rc = ctx_enter_device(m->ctx);
  if (rc) return rc;
  hipStream_t s = ctx_stream_of(m->ctx);
  const long chunk = 16384;
  if ((rc = ensure_work(m, (int)std::min(chunk, (n + 63) / 64 * 64)))) return rc;
  const int L = m->L;
  for (long r0 = 0; r0 < n; r0 += chunk) {
    const int nr = (int)std::min(chunk, n - r0);
    const int rows = (nr + 63) / 64 * 64;
    if ((rc = launch_rows_to_bf16(X_dev + r0 * ldx, ldx, nullptr, nr, rows, m->dims[0], m->X0,
                                  m->pad[0], s)) ||
        (rc = forward(m, rows, s)))
      return rc;
    BIHIP_HIP(hipMemcpy2DAsync(Y_dev + r0 * ldy, sizeof(float) * ldy, m->Z[L - 1],
                               sizeof(float) * m->pad[L], sizeof(float) * m->dims[L], nr,
                               hipMemcpyDeviceToDevice, s));
  }
  return BIHIP_OK;
}

int bihip_mlp_loss_grad(bihip_mlp* m, const float* X_dev, long ldx, const float* T_dev, long ldt,
                        int n, double* loss_host, float* grad_host) {
  if (m == nullptr || X_dev == nullptr || T_dev == nullptr)
    return set_error(BIHIP_EINVAL, "NULL argument");
  if (n <= 0 || ldx < m->dims[0] || ldt < targets_per_sample(m))
    return set_error(BIHIP_EINVAL, "bad n or leading dimensions");
  int rc = ctx_enter_device(m->ctx);
  if (rc) return rc;
  hipStream_t s = ctx_stream_of(m->ctx);
  const int rows = (n + 63) / 64 * 64;
  if ((rc = ensure_work(m, rows))) return rc;
  double sq = 0.0;
  if ((rc = launch_rows_to_bf16(X_dev, ldx, nullptr, n, rows, m->dims[0], m->X0, m->pad[0], s)) ||
      (rc = forward(m, rows, s)) ||
      (rc = loss_and_error(m, T_dev, ldt, nullptr, n, rows, &sq, s)) ||
      (rc = backward(m, rows, UpdateArgs{}, s)))
    return rc;
  if (loss_host) *loss_host = sq / ((double)n * targets_per_sample(m));
  if (grad_host) {
    std::vector<float> G(m->ntot);
    BIHIP_HIP(hipMemcpyAsync(G.data(), m->G, sizeof(float) * m->ntot, hipMemcpyDeviceToHost, s));
    BIHIP_HIP(hipStreamSynchronize(s));
    unpack(m, G, grad_host);
  }
  return BIHIP_OK;
}

int bihip_mlp_train(bihip_mlp* m, const float* X_dev, long ldx, const float* T_dev, long ldt,
                    long n, int batch, int steps, float lr, uint64_t seed, float* loss_host) {
  if (m == nullptr || X_dev == nullptr || T_dev == nullptr)
    return set_error(BIHIP_EINVAL, "NULL argument");
  if (ldt < targets_per_sample(m)) return set_error(BIHIP_EINVAL, "ldt below the targets per sample");
  if (n <= 0 || batch <= 0 || batch % 64 || batch > n || steps < 0 || !(lr > 0.0f))
    return set_error(BIHIP_EINVAL, "need 0 < batch <= n, batch a multiple of 64, lr > 0");
  int rc = ctx_enter_device(m->ctx);
  if (rc) return rc;
  hipStream_t s = ctx_stream_of(m->ctx);
  if ((rc = ensure_work(m, batch))) return rc;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  long* perm_d = nullptr;
  float* loss_d = nullptr;
  double* unif_d = nullptr;  // an epoch's uniforms
  if ((rc = dalloc(&perm_d, (size_t)n)) || (rc = dalloc(&loss_d, (size_t)std::max(steps, 1))) ||
      (rc = dalloc(&unif_d, (size_t)std::min(n, UNIF_CHUNK)))) {
    dfree(perm_d);
    dfree(loss_d);
    return rc;
  }
  std::vector<double> unif((size_t)std::min(n, UNIF_CHUNK));
  std::vector<long> perm(n);
  std::iota(perm.begin(), perm.end(), 0L);
  long pos = n;  // position in the current epoch's permutation
  long epoch = -1;
  for (int it = 0; it < steps && rc == BIHIP_OK; ++it) {
    if (pos + batch > n) {  // new epoch: Fisher-Yates with keyed uniforms
      ++epoch;
      // uniform i keyed by (seed, i, epoch), drawn on the device a chunk at a
      // time: on the host they took four fifths of the shuffle
      for (long hi = n; hi > 1 && rc == BIHIP_OK;) {
        const long lo = (hi - 1) / UNIF_CHUNK * UNIF_CHUNK;
        if ((rc = launch_uniforms_at(seed, lo, (uint32_t)epoch, TAG_MLP_BATCH, (int)(hi - lo),
                                     unif_d, s)))
          break;
        if (hipMemcpyAsync(unif.data(), unif_d, sizeof(double) * (hi - lo), hipMemcpyDeviceToHost,
                           s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess) {
          rc = set_error(BIHIP_EHIP, "reading the batch shuffle's uniforms failed");
          break;
        }
        for (long i = hi - 1; i >= std::max(lo, 1L); --i) {
          const long j = std::min(i, (long)(unif[i - lo] * (double)(i + 1)));
          std::swap(perm[i], perm[j]);
        }
        hi = lo;
      }
      if (rc != BIHIP_OK) break;
      // the previous epoch's batches must have read perm_d before it changes
      if (hipStreamSynchronize(s) != hipSuccess ||
          hipMemcpyAsync(perm_d, perm.data(), sizeof(long) * n, hipMemcpyHostToDevice, s) !=
              hipSuccess) {
        rc = set_error(BIHIP_EHIP, "uploading the batch permutation failed");
        break;
      }
      pos = 0;
    }
    const long* idx = perm_d + pos;
    pos += batch;
    int nb = 0;
    if ((rc = launch_rows_to_bf16(X_dev, ldx, idx, batch, batch, m->dims[0], m->X0, m->pad[0],
                                  s)) ||
        (rc = forward(m, batch, s)) ||
        (rc = output_error(m, T_dev, ldt, idx, batch, batch, &nb, s)))
      break;
    ++m->adam_t;
    UpdateArgs u{};
    u.adam = 1;
    u.lr = lr;
    u.b1 = b1;
    u.b2 = b2;
    u.eps = eps;
    u.bc1 = 1.0f - std::pow(b1, (float)m->adam_t);
    u.bc2 = 1.0f - std::pow(b2, (float)m->adam_t);
    u.loss = m->lossp;
    u.nloss = nb;
    u.loss_out = loss_d + it;
    if ((rc = backward(m, batch, u, s))) break;
  }
  if (rc == BIHIP_OK && loss_host != nullptr && steps > 0) {
    std::vector<float> h(steps);
    if (hipMemcpyAsync(h.data(), loss_d, sizeof(float) * steps, hipMemcpyDeviceToHost, s) !=
            hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      rc = set_error(BIHIP_EHIP, "reading the losses failed");
    const float inv = 1.0f / ((float)batch * (float)targets_per_sample(m));
    for (int it = 0; it < steps && rc == BIHIP_OK; ++it) loss_host[it] = h[it] * inv;
  }
  (void)hipStreamSynchronize(s);
  dfree(perm_d);
  dfree(loss_d);
  dfree(unif_d);
  return rc;
}

int bihip_mlp_set_loss(bihip_mlp* m, int loss) {
  if (m == nullptr) return set_error(BIHIP_EINVAL, "NULL network");
  if (loss != BIHIP_LOSS_MSE && loss != BIHIP_LOSS_GAUSS)
    return set_error(BIHIP_EINVAL, "unknown loss %d", loss);
  if (loss == BIHIP_LOSS_GAUSS && m->dims[m->L] % 2)
    return set_error(BIHIP_EINVAL, "the Gaussian loss needs an even output width");
  m->loss = loss;
  return BIHIP_OK;
}

int bihip_surrogate_flow(bihip_ctx* ctx, bihip_mlp* m, const bihip_surrogate_norm* norm,
                         double par, const float* Xin_dev, float* Xout_dev, int ld, int P) {
  int rc = ctx_enter_device(ctx);
  if (rc) return rc;
  if (m == nullptr || norm == nullptr || Xin_dev == nullptr || Xout_dev == nullptr)
    return set_error(BIHIP_EINVAL, "NULL argument");
  if (P < 0 || ld < P) return set_error(BIHIP_EINVAL, "need 0 <= P <= ld");
  if (Xin_dev == Xout_dev) return set_error(BIHIP_EINVAL, "the flow is out of place");
  SurrogateLaunch L{};
  L.net = mlp_view(m);
  if ((rc = mlp_inference_weights(m, ctx_stream_of(ctx), L.Winf, L.binf))) return rc;
  L.x_shift = norm->x_shift;
  L.x_scale = norm->x_scale;
  L.dx_scale = norm->dx_scale;
  L.par = par;
  L.par_shift = norm->par_shift;
  L.par_scale = norm->par_scale;
  L.Xin = Xin_dev;
  L.Xout = Xout_dev;
  L.ld = ld;
  L.P = P;
  L.step = false;
  if ((rc = launch_surrogate(L, ctx_stream_of(ctx)))) return rc;
  return note_reader(m, ctx_stream_of(ctx));
}

int bihip_guided_propose(bihip_ctx* ctx, bihip_mlp* m, const bihip_guided_norm* norm, double par,
                         float* X_dev, int ld, int P, const double* y_dev, uint64_t seed,
                         uint32_t batch, uint32_t step, double noise_sd, double obs_sd,
                         double* inc_dev) {
  int rc = ctx_enter_device(ctx);
  if (rc) return rc;
  if (m == nullptr || norm == nullptr || X_dev == nullptr || y_dev == nullptr || inc_dev == nullptr)
    return set_error(BIHIP_EINVAL, "NULL argument");
  if (P < 0 || ld < P) return set_error(BIHIP_EINVAL, "need 0 <= P <= ld");
  GuidedLaunch G{};
  G.net = mlp_view(m);
  if ((rc = mlp_inference_weights(m, ctx_stream_of(ctx), G.Winf, G.binf, 16))) return rc;
  G.x_shift = norm->x_shift;
  G.x_scale = norm->x_scale;
  G.innov_scale = norm->innov_scale;
  G.par = par;
  G.par_shift = norm->par_shift;
  G.par_scale = norm->par_scale;
  G.X = X_dev;
  G.ld = ld;
  G.P = P;
  G.y = y_dev;
  G.seed = seed;
  G.batch = batch;
  G.step = step;
  G.noise_sd = (float)noise_sd;
  G.obs_sd = obs_sd;
  G.inc = inc_dev;
  if ((rc = launch_guided(G, ctx_stream_of(ctx)))) return rc;
  return note_reader(m, ctx_stream_of(ctx));
}

}  // extern "C"
