// Fused predict + correct kernel: (ancestor gather) -> noise -> ODE flow ->
// observation log-density -> per-block weight partials.  One particle per
// lane group; state in registers; each state column is read and written
// once, coalesced across particles (structure-of-arrays).
//
// Replaces, for the ON_DEVICE location:
//   Model::transitionSamples       share/tt/cpp/model.hpp.tt:566-573
//   StaticSamplerHost::samples     share/src/bi/host/updater/StaticSamplerHost.hpp:43-65
//   RK4/DOPRI5IntegratorHost       share/src/bi/host/ode/{RK4,DOPRI5}IntegratorHost.hpp
//   observationLogDensities        share/src/bi/host/updater/SparseStaticLogDensityHost.hpp:46-68
//   gather_rows (fused read)       share/src/bi/host/primitive/matrix_primitive.hpp:65-75
#include <cstring>

#include "model_ops.hpp"
#include "blockreduce.hpp"
#include "internal.hpp"
#include "gen_model.hpp"

namespace bihip {

struct TransArgs {
  ModelArgs m;
  const void* Xin;
  void* Xout;
  int ld, P;
  const int* as;
  double* lws;
  const double* y;
  double t1, t2;
  uint64_t seed;
  uint32_t step, batch;
  int* nsteps_out;
  double* partials;
  const PFDevice* dev;
  double t0, dt;
  const double* y_base;
  int nobs;
  int flow_only;        // 1: deterministic flow, no noise (integrator update)
  const double* aux;    // flow_only: per-particle noise variable (PZ alpha) or null
  const double* times;  // with dev: schedule times (nullable: t0 + k dt)
  const int* mask;      // with dev: observed flags (nullable: every step observed)
  const double* inputs; // with dev: 16 model parameters per step (nullable)
  const int* imp_r;     // with dev: imposed resampling flags per step (nullable)
  BankStrides bk;       // BANK: strides of the filters (filter f = blockIdx.y)
  const double* bank_par;  // BANK: BANK_ROW parameters per filter
  void* noise_hist;     // SCHED, with dev (nullable): the step's noise variables into
                        // slot k + 1 of a (T + 1) x noise_width x ld history
  int noise_width;
};

// ---------------------------------------------------------------- the kernel
// A value the whole wave shares, moved to a scalar register so that the
// compiler keeps what derives from it out of vector registers.
__device__ __forceinline__ double uniform(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readfirstlane((int)b);
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// SCHED: the filter step has a schedule or inputs (times, observed flags,
// per-step parameters); without them the kernel is compiled without that code,
// which costs the plain step about 7% when present but unused.
// Waves per SIMD the compiler must leave room for: the functor names its own.
template <class M>
constexpr int trans_min_waves() {
  return M::MIN_WAVES;
}

// ONE: a generated model's interval is one sub-interval of its delta that
// starts at a multiple of it (its transition runs without the sub-interval loop).
// BANK: filter blockIdx.y of a bank, with its own state, vectors, PFDevice,
// Philox batch id and parameter row (then the step is exactly a lone
// filter's with those parameters and that batch id).
template <class M, int INTEG, bool SCHED = false, bool ONE = false, bool BANK = false>
__global__ __launch_bounds__(TRANS_BLOCK) __attribute__((amdgpu_waves_per_eu(trans_min_waves<M>())))
void k_transition(TransArgs a) {
  using T = typename M::real_t;
  constexpr int LPP = M::LPP, DL = M::DL;
  if constexpr (BANK) {
    const long f = blockIdx.y;
    a.Xin = bank_shift(a.Xin, f * a.bk.x * (long)sizeof(T));
    a.Xout = bank_shift(a.Xout, f * a.bk.x * (long)sizeof(T));
    a.as = bank_shift(a.as, f * a.bk.p * (long)sizeof(int));
    a.lws = bank_shift(a.lws, f * a.bk.p * (long)sizeof(double));
    a.partials = bank_shift(a.partials, f * (long)gridDim.x * 3 * (long)sizeof(double));
    a.dev = a.dev + f;
    a.batch += (uint32_t)f;
    const double* row = a.bank_par + BANK_ROW * f;
#pragma unroll
    for (int i = 0; i < 16; ++i) a.m.par[i] = uniform(row[i]);
    a.m.obs_inv = uniform(row[16]);
    a.m.obs_c = uniform(row[17]);
  }
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const int p = blk * (TRANS_BLOCK / LPP) + (int)threadIdx.x / LPP;
  const Group<LPP> grp;
  const int lo = slice_lo<M>(grp.g);
  const bool active = p < a.P;

  bool gather = a.as != nullptr;
  bool lws_const = false;
  double lws_base = 0.0;
  double t1 = a.t1, t2 = a.t2;
  uint32_t step = a.step;
  const double* y = a.y;
  // the inputs in force over [t_k, t_{k+1}) (Forcer): the step's parameters
  const double* in = SCHED && a.dev != nullptr && a.inputs != nullptr
                         ? a.inputs + (size_t)16 * a.dev->k
                         : nullptr;
  if (a.dev != nullptr) {
    const int k = a.dev->k;
    gather = a.imp_r != nullptr ? a.imp_r[k] != 0
                                : a.dev->resample != 0 && a.dev->status == BIHIP_OK;
    lws_const = gather;
    lws_base = a.dev->logLikelihood;
    t1 = SCHED && a.times != nullptr ? a.times[k] : a.t0 + k * a.dt;
    t2 = SCHED && a.times != nullptr ? a.times[k + 1] : a.t0 + (k + 1) * a.dt;
    step = (uint32_t)(k + 1);
    // BootstrapPF::correct applies only at observed elements
    // (share/src/bi/filter/BootstrapPF.hpp:171-181); null y_base: flow only
    const bool observed = !SCHED || a.mask == nullptr || a.mask[k] != 0;
    y = a.y_base != nullptr && observed ? a.y_base + (size_t)k * a.nobs : nullptr;
  }

  double lw = __builtin_nan("");
  if (active) {
    const int src = gather ? a.as[p] : p;
    const T* Xin = static_cast<const T*>(a.Xin);
    T x[DL];
#pragma unroll
    for (int i = 0; i < DL; ++i)
      x[i] = slice_has<M>(grp.g, i) ? Xin[(size_t)(lo + i) * a.ld + src] : T(0);

    auto model = [&]() {
      if (!SCHED || in == nullptr) return M(a.m);
      ModelArgs ma = a.m;
#pragma unroll
      for (int i = 0; i < 16; ++i) ma.par[i] = uniform(in[i]);
      return M(ma);
    };
    M m = model();
    int n;
    T* zout = nullptr;  // the noise variables of this step (recorded histories only)
    if constexpr (SCHED) {
      if (a.noise_hist != nullptr && a.dev != nullptr && !a.flow_only)
        zout = static_cast<T*>(a.noise_hist) +
               (size_t)(a.dev->k + 1) * (size_t)a.noise_width * (size_t)a.ld;
    }
    if constexpr (is_generated<M>::value) {
      // the model's transition block: discrete actions and its ode, in order
      n = m.template transition<INTEG, ONE>(grp, x, t1, t2, a.m, a.seed, a.batch, (uint32_t)p,
                                            step);
      if constexpr (SCHED) {
        if (zout != nullptr) m.noise_out(grp, zout, a.ld, (uint32_t)p);
      }
    } else {
      if constexpr (M::NOISE_FIRST) {
        if (!a.flow_only) {
          noise_first(m, a.seed, a.batch, p, step);
          if (SCHED && zout != nullptr && grp.g == 0) zout[p] = m.alpha;  // PZ's alpha
        } else {
          m.alpha = a.aux != nullptr ? (T)a.aux[p] : (T)m.mu;
        }
      }
      if constexpr (INTEG == BIHIP_RK4) {
        n = integrate_rk4(m, grp, x, t1, t2, a.m.h0);
      } else {
        n = integrate_dopri5(m, grp, x, t1, t2, a.m);
      }
      if constexpr (!M::NOISE_FIRST) {
        if (!a.flow_only) noise_after(m, a.seed, a.batch, p, lo, step, x, zout, a.ld);
      }
    }

    T* Xout = static_cast<T*>(a.Xout);
#pragma unroll
    for (int i = 0; i < DL; ++i)
      if (slice_has<M>(grp.g, i)) Xout[(size_t)(lo + i) * a.ld + p] = x[i];
    if (a.nsteps_out != nullptr && grp.g == 0) a.nsteps_out[p] = n;

    if (y != nullptr) {
      // observation constants from the host, or from the step's inputs
      const double part =
          grp.sum(obs_of(m, x, y, lo, !SCHED || in == nullptr ? &a.m : nullptr));
      if (grp.g == 0) {
        const double base = lws_const ? lws_base : a.lws[p];
        lw = base + part;
        a.lws[p] = lw;
      }
    } else if (SCHED && lws_const && a.lws != nullptr && grp.g == 0) {
      a.lws[p] = lws_base;  // resampled, then no observation: lws = logLikelihood
    }
  }
  // only group leaders (lanes g == 0) hold a log-weight
  if constexpr (!uneven_slices<M>()) {
    if (a.partials != nullptr)
      block_weight_partial<TRANS_BLOCK, LPP>(lw, a.partials + 3 * blk);
  }
}

// Weight partials of PAIR_PARTIAL particles from the log-weights, one particle a
// lane, for models of which a pair of lanes holds one slice: their workgroups hold
// half a partial's particles.  Sums in the order of a workgroup with a lane per
// slice (waves of eight particles: a butterfly, then the four waves), whatever
// the lanes of a particle, so that log-likelihoods and effective sample sizes keep
// their bits.  3 us; workgroups of 512 threads, which hold a partial's particles,
// run two waves per SIMD where the registers allow three (a bank of 16 x 16384
// filters over five intervals 2.84 ms against 1.85).
constexpr int PAIR_PARTIAL = 32;

__global__ __launch_bounds__(256) void k_pair_partials(const double* lws, int P,
                                                       double* partials, int nb,
                                                       BankStrides bk) {
  const long f = blockIdx.y;
  lws = bank_shift(lws, f * bk.p * (long)sizeof(double));
  partials += 3 * f * nb;
  const int p = blockIdx.x * 256 + (int)threadIdx.x;
  const double lw = p < P ? lws[p] : __builtin_nan("");
  auto add = [](double x, double y) { return x + y; };
  auto larger = [](double x, double y) { return nan_max(x, y); };
  double m = xor_step<1>(lw, larger);
  m = xor_step<2>(m, larger);
  m = xor_step<4>(m, larger);
  m = xor_step<8>(m, larger);
  m = xor_step<16>(m, larger);
  const double z = nanexp(lw - m);
  double s1 = xor_step<1>(z, add);
  double s2 = fused(z, z, dpp<QP_XOR1>(z * z));
  s1 = xor_step<4>(xor_step<2>(s1, add), add);
  s2 = xor_step<4>(xor_step<2>(s2, add), add);
  const int first = (int)threadIdx.x & (WAVE - PAIR_PARTIAL);  // lane of the partial's first
  double t1 = __shfl(s1, first, WAVE), t2 = __shfl(s2, first, WAVE);
#pragma unroll
  for (int i = 8; i < PAIR_PARTIAL; i += 8) {
    t1 += __shfl(s1, first + i, WAVE);
    t2 += __shfl(s2, first + i, WAVE);
  }
  if (p % PAIR_PARTIAL == 0 && p < P) {
    double* out = partials + 3 * (p / PAIR_PARTIAL);
    out[0] = m;
    out[1] = t1;
    out[2] = t2;
  }
}

// ---------------------------------------------------------------- initial states
// bank_par (nullable): filter blockIdx.y of a bank, parameter row
// bank_par + BANK_ROW y, batch id batch + y, state at Xv + y * bx elements.
template <class M>
__global__ __launch_bounds__(TRANS_BLOCK) void k_init(ModelArgs ma, uint64_t seed,
                                                      uint32_t batch, int P, void* Xv, int ld,
                                                      const double* mean0,
                                                      const double* bank_par, long bx) {
  using T = typename M::real_t;
  constexpr int LPP = M::LPP, DL = M::DL;
  if (bank_par != nullptr) {
    const long f = blockIdx.y;
    const double* row = bank_par + BANK_ROW * f;
    for (int i = 0; i < 16; ++i) ma.par[i] = row[i];
    ma.obs_inv = row[16];
    ma.obs_c = row[17];
    batch += (uint32_t)f;
    Xv = bank_shift(Xv, f * bx * (long)sizeof(T));
  }
  const int p = blockIdx.x * (TRANS_BLOCK / LPP) + (int)threadIdx.x / LPP;
  const Group<LPP> grp;
  const int lo = slice_lo<M>(grp.g);
  if (p >= P) return;
  T* X = static_cast<T*>(Xv);
  if constexpr (is_generated<M>::value) {
    double xd[DL];
    M(ma).init(xd, seed, batch, (uint32_t)p, lo);
#pragma unroll
    for (int i = 0; i < DL; ++i) X[(size_t)(lo + i) * ld + p] = (T)xd[i];
    return;
  }
  T z[DL];
  slice_normals<T, DL>(seed, (uint32_t)p, 0, TAG_INIT, batch, lo, z);
#pragma unroll
  for (int i = 0; i < DL; ++i) {
    double v;
    if (ma.model == BIHIP_MODEL_PZ) {
      v = i == 0 ? exp(ma.par[7] + ma.par[8] * (double)z[0])
                 : exp(ma.par[9] + ma.par[10] * (double)z[1]);
    } else if (ma.model == BIHIP_MODEL_L96) {
      if (!slice_has<M>(grp.g, i)) break;
      v = mean0[lo + i] + ma.par[3] * (double)z[i];
    } else {
      v = ma.par[3] + ma.par[4] * (double)z[i];
    }
    X[(size_t)(lo + i) * ld + p] = (T)v;
  }
}

// ---------------------------------------------------------------- standalone correction
template <class M>
__global__ __launch_bounds__(TRANS_BLOCK) void k_obs_logdensity(ModelArgs ma, const double* y,
                                                                int P, const void* Xv, int ld,
                                                                double* lws) {
  using T = typename M::real_t;
  constexpr int LPP = M::LPP, DL = M::DL;
  const int p = blockIdx.x * (TRANS_BLOCK / LPP) + (int)threadIdx.x / LPP;
  const Group<LPP> grp;
  const int lo = slice_lo<M>(grp.g);
  if (p >= P) return;
  const T* X = static_cast<const T*>(Xv);
  T x[DL];
#pragma unroll
  for (int i = 0; i < DL; ++i)
    x[i] = slice_has<M>(grp.g, i) ? X[(size_t)(lo + i) * ld + p] : T(0);
  M m(ma);
  const double part = grp.sum(obs_of(m, x, y, lo));
  if (grp.g == 0) lws[p] = lws[p] + part;
}

// Observation samples (Model::observationSamples), y is P x nobs.
template <class M>
__global__ __launch_bounds__(TRANS_BLOCK) void k_obs_sample(ModelArgs ma, uint64_t seed,
                                                            uint32_t batch, uint32_t step, int P,
                                                            const void* Xv, int ld, double* y) {
  using T = typename M::real_t;
  const int p = blockIdx.x * TRANS_BLOCK + threadIdx.x;
  if (p >= P) return;
  const T* X = static_cast<const T*>(Xv);
  constexpr int NOBS = M::NOBS;
  if constexpr (is_generated<M>::value) {  // the whole state of the particle
    T x[M::D];
#pragma unroll
    for (int i = 0; i < M::D; ++i) x[i] = X[(size_t)i * ld + p];
    double yo[NOBS > 0 ? NOBS : 1];
    M(ma).obs_sample(x, seed, batch, (uint32_t)p, step, yo);
    for (int o = 0; o < NOBS; ++o) y[(size_t)p * NOBS + o] = yo[o];
    return;
  }
  for (int b = 0; 4 * b < NOBS; ++b) {
    T z[4];
    normals4<T>(seed, (uint32_t)p, step, TAG_OBS, batch, (uint32_t)b, z);
    for (int i = 0; i < 4 && 4 * b + i < NOBS; ++i) {
      const int o = 4 * b + i;
      double v;
      if (ma.model == BIHIP_MODEL_PZ) {
        v = exp(log((double)X[p]) + ma.par[6] * (double)z[i]);
      } else if (ma.model == BIHIP_MODEL_L96) {
        v = (double)X[(size_t)(2 * o) * ld + p] + ma.par[2] * (double)z[i];
      } else {
        v = (double)X[p] + ma.par[2] * (double)z[i];
      }
      y[(size_t)p * NOBS + o] = v;
    }
  }
}

// ---------------------------------------------------------------- random-number utilities
__global__ void k_philox(const uint32_t* ctr, uint32_t k0, uint32_t k1, int n, uint32_t* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const u32x4 r = philox4x32_10(ctr[4 * i], ctr[4 * i + 1], ctr[4 * i + 2], ctr[4 * i + 3], k0, k1);
  out[4 * i] = r.x;
  out[4 * i + 1] = r.y;
  out[4 * i + 2] = r.z;
  out[4 * i + 3] = r.w;
}

__global__ void k_uniforms(uint64_t seed, uint32_t step, uint32_t tag, uint32_t batch, int n,
                           double* u) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const u32x4 r = philox_block(seed, (uint32_t)j, step, tag, batch, 0);
  u[j] = u53(r.x, r.y);
}

// u[j] of index base + j, its high word as the batch id
__global__ void k_uniforms_at(uint64_t seed, long base, uint32_t step, uint32_t tag, int n,
                              double* u) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const long i = base + j;
  const u32x4 r = philox_block(seed, (uint32_t)i, step, tag, (uint32_t)(i >> 32), 0);
  u[j] = u53(r.x, r.y);
}

template <class T>
__global__ void k_normals(uint64_t seed, uint32_t index, uint32_t step, uint32_t tag,
                          uint32_t batch, int n, T* z) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (4 * b >= n) return;
  T q[4];
  normals4<T>(seed, index, step, tag, batch, (uint32_t)b, q);
  for (int i = 0; i < 4 && 4 * b + i < n; ++i) z[4 * b + i] = q[i];
}

// ---------------------------------------------------------------- dispatch
const GenInfo* generated_info(int model) {
  const int i = model - BIHIP_MODEL_GENERATED;
  return i >= 0 && i < GEN_COUNT ? &GEN_MODELS[i] : nullptr;
}

bool model_supported(const bihip_model* m) {
  if (m->integrator != BIHIP_RK4 && m->integrator != BIHIP_DOPRI5) return false;
  if (m->precision != BIHIP_F32 && m->precision != BIHIP_F64) return false;
  if (const GenInfo* g = generated_info(m->model)) return m->d == g->d;
  switch (m->model) {
    case BIHIP_MODEL_PZ: return m->d == 2;
    case BIHIP_MODEL_L96: return m->d == 8 || m->d == 40 || m->d == 200;
    case BIHIP_MODEL_LG: return m->d == 1;
  }
  return false;
}

// Lanes per particle of the Lorenz-96 d=40 model.  Four: ten dimensions per
// lane, 112 VGPRs.  Two lanes (twenty dimensions each, ten Philox blocks per
// particle instead of twelve) need 216 VGPRs, two waves per SIMD, and
// measured 234 us per N = 2^20 FP32 transition against 207-210 us.
#ifndef L96_D40_LPP
#define L96_D40_LPP 4
#endif
// d = 200: eight lanes of 25 dimensions or sixteen of 13 and 12 (a DPP row), the
// same bits.  Sixteen need fewer registers (FP32 DOPRI5 138 against 246, FP64 256
// with 12 bytes of spills against 512 with 260) and no LDS permutes for the halos,
// and half the steps' latency; but a wave's load or store of a row spans four
// particles, 16 bytes in FP32, which costs more where memory bounds.  us per
// transition, eight / sixteen lanes, of
//                       1000         8192         30000        262144 particles
//   FP32 DOPRI5         15.4 / 10.2  16.4 / 15.4  35.9 / 41.9   254 / 289
//   FP32 RK4, 5 steps   12.4 /  8.7  13.4 / 13.3  26.5 / 33.5   189 / 246
//   FP64 DOPRI5         28.9 / 15.0  31.7 / 25.5   117 / 81     964 / 672
//   FP64 RK4, 1 step    12.3 /  8.6  15.0 / 14.5  38.6 / 36.1   336 / 368
//   FP64 RK4, 5 steps   17.3 / 11.5  19.9 / 19.5  52.3 / 53.9   409 / 437
// so FP32 takes sixteen up to 8192 particles, FP64 always but for RK4 above 2^16
// (60000 particles, five steps: 96.1 / 94.4).  A bank's FP32 DOPRI5 kernel takes
// sixteen too: with eight its 273 registers leave one wave per SIMD (16 x 16384
// filters over five intervals 2.85 ms, with sixteen 1.85).
static bool d200_sixteen_lanes(const bihip_model* m, long particles, bool bank) {
  const bool rk4 = m->integrator == BIHIP_RK4;
  if (m->precision == BIHIP_F32) return particles <= 8192 || (bank && !rk4);
  return !rk4 || particles <= 1L << 16;
}

// Calls F::template run<M>() for the model type selected by m (sixteen: d = 200
// over sixteen lanes).
template <class F>
static int with_model(const bihip_model* m, F& f, bool sixteen = false) {
  const bool f64 = m->precision == BIHIP_F64;
  if (m->model >= BIHIP_MODEL_GENERATED) return with_generated(m, f);
  switch (m->model) {
    case BIHIP_MODEL_PZ:
      return f64 ? f.template run<PZ<double>>() : f.template run<PZ<float>>();
    case BIHIP_MODEL_L96:
      if (m->d == 40)
        return f64 ? f.template run<L96<double, 40, L96_D40_LPP>>()
                   : f.template run<L96<float, 40, L96_D40_LPP>>();
      if (m->d == 200)
        return sixteen ? (f64 ? f.template run<L96<double, 200, 16>>()
                              : f.template run<L96<float, 200, 16>>())
                       : (f64 ? f.template run<L96<double, 200, 8>>()
                              : f.template run<L96<float, 200, 8>>());
      return f64 ? f.template run<L96<double, 8, 2>>() : f.template run<L96<float, 8, 2>>();
    default:
      return f64 ? f.template run<LG<double>>() : f.template run<LG<float>>();
  }
}

// Workgroups of model M's kernels.
template <class M>
static int model_blocks(int P) {
  return ceil_div((long)P * M::LPP, TRANS_BLOCK);
}

int transition_blocks(const bihip_model* m, int P) {
  int lpp = 1;
  if (m->model == BIHIP_MODEL_L96) lpp = m->d == 200 ? 8 : (m->d == 40 ? L96_D40_LPP : 2);
  if (const GenInfo* g = generated_info(m->model)) lpp = g->lpp;
  return ceil_div((long)P * lpp, TRANS_BLOCK);
}

// [t1, t2] is one sub-interval of delta starting at a multiple of it, with a
// margin (1e-6 of delta) far inside the device's rounding window (1e-4,
// gen_scaled), so that the device's own rounding of t1 and t2 decides alike.
static bool one_interval(double t1, double t2, double delta) {
  const double s1 = t1 / delta, s2 = t2 / delta;
  const double r1 = std::round(s1), r2 = std::round(s2);
  return std::fabs(s1 - r1) < 1e-6 && std::fabs(s2 - r2) < 1e-6 && r2 == r1 + 1.0;
}

bool gen_one_delta(const bihip_model* m, double t0, double dt, int steps) {
  const GenInfo* g = generated_info(m->model);
  if (g == nullptr || steps <= 0) return false;
  for (int k = 0; k < steps; ++k)
    if (!one_interval(t0 + k * dt, t0 + (k + 1) * dt, g->delta)) return false;
  return true;
}

struct TransitionRunner {
  TransArgs a;
  hipStream_t s;
  int integ;
  bool one;
  int banks;
  template <class M>
  int run() {
    const int rc = run_transition<M>();
    if constexpr (uneven_slices<M>()) {
      if (rc == BIHIP_OK && a.partials != nullptr) {
        hipLaunchKernelGGL(k_pair_partials, dim3(ceil_div(a.P, 256), banks > 1 ? banks : 1),
                           dim3(256), 0, s, (const double*)a.lws, a.P, a.partials,
                           ceil_div(a.P, PAIR_PARTIAL), a.bk);
        BIHIP_LAUNCH_CHECK();
      }
    }
    return rc;
  }
  template <class M>
  int run_transition() {
    const int blocks = model_blocks<M>(a.P);
    const bool sched = a.dev != nullptr && (a.times != nullptr || a.mask != nullptr ||
                                            a.inputs != nullptr || a.noise_hist != nullptr);
    if (banks > 1 || a.bank_par != nullptr) {  // a bank, also of one filter: its rows
      // a generated model runs its general interval loop over delta (the
      // one-delta form gives the same values)
      if (sched || a.dev == nullptr || a.bank_par == nullptr || a.imp_r != nullptr)
        return set_error(BIHIP_EINVAL, "a filter bank step takes no schedule, inputs or "
                                       "imposed history");
      const dim3 grid(blocks, banks > 1 ? banks : 1);
      if (integ == BIHIP_RK4)
        hipLaunchKernelGGL((k_transition<M, BIHIP_RK4, false, false, true>), grid,
                           dim3(TRANS_BLOCK), 0, s, a);
      else
        hipLaunchKernelGGL((k_transition<M, BIHIP_DOPRI5, false, false, true>), grid,
                           dim3(TRANS_BLOCK), 0, s, a);
      BIHIP_LAUNCH_CHECK();
      return BIHIP_OK;
    }
    if constexpr (is_generated<M>::value) {
      if (one && !sched) {
        if (integ == BIHIP_RK4)
          hipLaunchKernelGGL((k_transition<M, BIHIP_RK4, false, true>), dim3(blocks),
                             dim3(TRANS_BLOCK), 0, s, a);
        else
          hipLaunchKernelGGL((k_transition<M, BIHIP_DOPRI5, false, true>), dim3(blocks),
                             dim3(TRANS_BLOCK), 0, s, a);
        BIHIP_LAUNCH_CHECK();
        return BIHIP_OK;
      }
    }
    if (integ == BIHIP_RK4) {
      if (sched)
        hipLaunchKernelGGL((k_transition<M, BIHIP_RK4, true>), dim3(blocks), dim3(TRANS_BLOCK), 0,
                           s, a);
      else
        hipLaunchKernelGGL((k_transition<M, BIHIP_RK4>), dim3(blocks), dim3(TRANS_BLOCK), 0, s, a);
    } else {
      if (sched)
        hipLaunchKernelGGL((k_transition<M, BIHIP_DOPRI5, true>), dim3(blocks), dim3(TRANS_BLOCK),
                           0, s, a);
      else
        hipLaunchKernelGGL((k_transition<M, BIHIP_DOPRI5>), dim3(blocks), dim3(TRANS_BLOCK), 0, s,
                           a);
    }
    BIHIP_LAUNCH_CHECK();
    return BIHIP_OK;
  }
};

int launch_transition(const TransLaunch& L, hipStream_t s) {
  if (L.P <= 0) return BIHIP_OK;
  TransitionRunner r;
  r.a.m = to_args(L.model);
  r.a.Xin = L.Xin;
  r.a.Xout = L.Xout;
  r.a.ld = L.ld;
  r.a.P = L.P;
  r.a.as = L.as;
  r.a.lws = L.lws;
  r.a.y = L.y;
  r.a.t1 = L.t1;
  r.a.t2 = L.t2;
  r.a.seed = L.seed;
  r.a.step = L.step;
  r.a.batch = L.batch;
  r.a.nsteps_out = L.nsteps_out;
  r.a.partials = L.partials;
  r.a.dev = L.dev;
  r.a.t0 = L.t0;
  r.a.dt = L.dt;
  r.a.times = L.times;
  r.a.mask = L.mask;
  r.a.inputs = L.inputs;
  r.a.y_base = L.y_base;
  r.a.nobs = L.nobs;
  r.a.flow_only = L.flow_only;
  r.a.aux = L.aux;
  r.a.imp_r = L.imp_r;
  r.a.bk = L.bk;
  r.a.bank_par = L.bank_par;
  r.a.noise_hist = L.noise_hist;
  r.a.noise_width = L.noise_width;
  r.banks = L.banks;
  r.s = s;
  r.integ = L.model->integrator;
  if (const GenInfo* g = generated_info(L.model->model))
    r.one = L.dev != nullptr ? L.one_delta != 0 : one_interval(L.t1, L.t2, g->delta);
  else
    r.one = false;
  return with_model(L.model, r,
                    d200_sixteen_lanes(L.model, (long)L.P * (L.banks > 1 ? L.banks : 1),
                                       L.bank_par != nullptr));
}

struct InitRunner {
  ModelArgs ma;
  uint64_t seed;
  uint32_t batch;
  int P, ld;
  void* X;
  const double* mean0;
  hipStream_t s;
  int banks;
  const double* bank_par;
  long bx;
  template <class M>
  int run() {
    hipLaunchKernelGGL((k_init<M>), dim3(model_blocks<M>(P), banks), dim3(TRANS_BLOCK), 0, s, ma, seed, batch,
                       P, X, ld, mean0, bank_par, bx);
    BIHIP_LAUNCH_CHECK();
    return BIHIP_OK;
  }
};

int launch_init_samples(const bihip_model* m, uint64_t seed, uint32_t batch, int P, void* X,
                        int ld, const double* mean0_dev, hipStream_t s) {
  if (P <= 0) return BIHIP_OK;
  InitRunner r{to_args(m), seed, batch, P, ld, X, mean0_dev, s,
               1, nullptr, 0};
  return with_model(m, r);
}

int launch_init_bank(const bihip_model* m, uint64_t seed, uint32_t batch, int P, void* X, int ld,
                     const double* mean0_dev, int banks, long x, const double* bank_par,
                     hipStream_t s) {
  if (P <= 0 || banks <= 0) return BIHIP_OK;
  InitRunner r{to_args(m), seed, batch, P, ld, X, mean0_dev, s,
               banks, bank_par, x};
  return with_model(m, r);
}

int noise_width_of(const bihip_model* m) {
  if (const GenInfo* g = generated_info(m->model)) {  // the model file's noise variables
    int w = 0;
    for (int i = 0; g->names[BIHIP_VAR_NOISE][i] != nullptr; ++i) w += g->sizes[BIHIP_VAR_NOISE][i];
    return w;
  }
  switch (m->model) {
    case BIHIP_MODEL_PZ: return 1;    // alpha
    case BIHIP_MODEL_L96: return m->d;  // w[n]
    default: return 1;                // w
  }
}

void bank_row(const bihip_model* m, double* row) {
  const ModelArgs a = to_args(m);
  for (int i = 0; i < 16; ++i) row[i] = a.par[i];
  row[16] = a.obs_inv;
  row[17] = a.obs_c;
}

struct ObsRunner {
  ModelArgs ma;
  const double* y;
  int P, ld;
  const void* X;
  double* lws;
  hipStream_t s;
  template <class M>
  int run() {
    hipLaunchKernelGGL((k_obs_logdensity<M>), dim3(model_blocks<M>(P)), dim3(TRANS_BLOCK), 0, s, ma, y, P, X,
                       ld, lws);
    BIHIP_LAUNCH_CHECK();
    return BIHIP_OK;
  }
};

int launch_obs_logdensity(const bihip_model* m, const double* y, int P, const void* X, int ld,
                          double* lws, hipStream_t s) {
  if (P <= 0) return BIHIP_OK;
  ObsRunner r{to_args(m), y, P, ld, X, lws, s};
  return with_model(m, r);
}

struct ObsSampleRunner {
  ModelArgs ma;
  uint64_t seed;
  uint32_t batch, step;
  int P, ld;
  const void* X;
  double* y;
  hipStream_t s;
  template <class M>
  int run() {
    hipLaunchKernelGGL((k_obs_sample<M>), dim3(ceil_div(P, TRANS_BLOCK)), dim3(TRANS_BLOCK), 0, s,
                       ma, seed, batch, step, P, X, ld, y);
    BIHIP_LAUNCH_CHECK();
    return BIHIP_OK;
  }
};

int launch_obs_sample(const bihip_model* m, uint64_t seed, uint32_t batch, uint32_t step, int P,
                      const void* X, int ld, double* y, hipStream_t s) {
  if (P <= 0) return BIHIP_OK;
  ObsSampleRunner r{to_args(m), seed, batch, step, P, ld, X, y, s};
  return with_model(m, r);
}

int launch_philox(const uint32_t* ctr, uint32_t k0, uint32_t k1, int n, uint32_t* out,
                  hipStream_t s) {
  if (n <= 0) return BIHIP_OK;
  hipLaunchKernelGGL(k_philox, dim3(ceil_div(n, 256)), dim3(256), 0, s, ctr, k0, k1, n, out);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_uniforms(uint64_t seed, uint32_t step, uint32_t tag, uint32_t batch, int n, double* u,
                    hipStream_t s) {
  if (n <= 0) return BIHIP_OK;
  hipLaunchKernelGGL(k_uniforms, dim3(ceil_div(n, 256)), dim3(256), 0, s, seed, step, tag, batch,
                     n, u);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_uniforms_at(uint64_t seed, long base, uint32_t step, uint32_t tag, int n, double* u,
                       hipStream_t s) {
  if (n <= 0) return BIHIP_OK;
  hipLaunchKernelGGL(k_uniforms_at, dim3(ceil_div(n, 256)), dim3(256), 0, s, seed, base, step, tag,
                     n, u);
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

int launch_normals(uint64_t seed, uint32_t index, uint32_t step, uint32_t tag, uint32_t batch,
                   int n, int precision, void* z, hipStream_t s) {
  if (n <= 0) return BIHIP_OK;
  const int nb = ceil_div(n, 4);
  if (precision == BIHIP_F64) {
    hipLaunchKernelGGL(k_normals<double>, dim3(ceil_div(nb, 256)), dim3(256), 0, s, seed, index,
                       step, tag, batch, n, static_cast<double*>(z));
  } else {
    hipLaunchKernelGGL(k_normals<float>, dim3(ceil_div(nb, 256)), dim3(256), 0, s, seed, index,
                       step, tag, batch, n, static_cast<float*>(z));
  }
  BIHIP_LAUNCH_CHECK();
  return BIHIP_OK;
}

}  // namespace bihip

using namespace bihip;

int bihip_model_generated(const char* name, int precision, bihip_model* m) {
  if (name == nullptr || m == nullptr) return set_error(BIHIP_EINVAL, "NULL argument");
  if (precision != BIHIP_F32 && precision != BIHIP_F64)
    return set_error(BIHIP_EINVAL, "precision must be BIHIP_F32 or BIHIP_F64");
  for (int i = 0; i < GEN_COUNT; ++i) {
    const GenInfo& g = GEN_MODELS[i];
    if (std::strcmp(g.name, name) != 0) continue;
    *m = bihip_model{};
    m->model = BIHIP_MODEL_GENERATED + i;
    m->d = g.d;
    m->integrator = g.integrator;
    m->nsteps = 1000;
    m->host_quirk = 0;
    m->precision = precision;
    m->h0 = g.h;
    m->atol = g.atol;
    m->rtol = g.rtol;
    return BIHIP_OK;
  }
  return set_error(BIHIP_EINVAL, "no generated model named '%s'", name);
}

const char* bihip_model_var_name(const bihip_model* m, int kind, int i) {
  const GenInfo* g = m ? generated_info(m->model) : nullptr;
  if (g == nullptr || i < 0 || kind < 0 || kind > 4) return nullptr;
  const char* const* names = g->names[kind];
  for (int k = 0; k <= i; ++k)
    if (names[k] == nullptr) return nullptr;
  return names[i];
}

int bihip_model_var_size(const bihip_model* m, int kind, int i) {
  return bihip_model_var_name(m, kind, i) != nullptr ? generated_info(m->model)->sizes[kind][i] : 0;
}

const char* bihip_model_name(const bihip_model* m) {
  const GenInfo* g = m ? generated_info(m->model) : nullptr;
  return g ? g->name : nullptr;
}
