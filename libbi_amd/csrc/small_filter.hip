// Whole steps of one small filter in one workgroup: BootstrapPF::step
// (share/src/bi/filter/BootstrapPF.hpp:156-167) for n observation intervals in
// one launch.
//
// A filter of at most 1024 particles leaves the chip idle whatever its kernels
// do: its step is the latency of its dependent launches.  Here one workgroup,
// one particle a thread, runs the resampling chain (small_chain.hpp), the
// gathered transition, the observation density, the weight partials and the
// bookkeeping of a step, and goes on to the next; the log-weights, the log-
// likelihood and the resampling decision stay in registers between steps.  Every
// sum keeps the order of the separate kernels (partials of 256 particles, then
// the combination's butterfly), so results equal theirs bit for bit.
//
// Bound by the latency of a step's arithmetic on one CU, and above 512 particles
// by its FP64 rate: up to four waves share a SIMD, where the separate launches
// give each wave its own.  Predator-prey filter (ten RK4 steps an interval) in
// FP64: 6.5 us a step at 200 particles, 9.0 at 500, 14.8 at 1000, against 12.2,
// 13.9 and 15.5 us in three launches (18 to 20 as graphs).  Long intervals turn
// this round above 256 particles (100 RK4 steps at 1000: 53.9 against 32 us), so
// small_filter_fits weighs the interval.  One particle a thread: up to 1024.
#include <cmath>

#include "blockreduce.hpp"
#include "gen_model.hpp"
#include "internal.hpp"
#include "model_ops.hpp"
#include "small_chain.hpp"

namespace bihip {

struct SmallFilterArgs {
  ModelArgs m;
  void* X[2];  // X[0]: the current state
  int ld, P, steps, resampler, nobs;
  int* as;
  double* lws;
  PFDevice* dev;
  PFHistory hist;
  const double* y;
  double t0, dt, essRel;
  uint64_t seed;
  uint32_t batch;
};

// Models it is compiled for: one lane per particle, few states (the workgroup
// leaves 128 registers a thread).
template <class M>
constexpr bool small_filter_model() {
  return M::LPP == 1 && M::D <= 4;
}

template <class M, int INTEG>
__global__ __launch_bounds__(SMALL_BLOCK) void k_filter_small(SmallFilterArgs a) {
  using T = typename M::real_t;
  constexpr int DL = M::DL, NB = SMALL_BLOCK / TRANS_BLOCK, WPB = TRANS_BLOCK / WAVE;
  static_assert(NB == 4 && WPB == 4, "a quad of lanes combines the partials");
  __shared__ SmallChainLds<1, true> chain;
  // the waves' maxima, in two buffers in turn: the last reads of a step's maxima
  // and the writes of the next one's have no barrier between them in a step that
  // does not resample (the sums' have the maxima's)
  __shared__ double wmax[2][SMALL_BLOCK / WAVE];
  __shared__ double w1[SMALL_BLOCK / WAVE], w2[SMALL_BLOCK / WAVE];
  const int p = threadIdx.x, lane = p & (WAVE - 1), w = p / WAVE;
  const bool active = p < a.P;
  const int nb = (a.P + TRANS_BLOCK - 1) / TRANS_BLOCK;
  const Group<1> grp;

  int k = a.dev->k, status = a.dev->status;
  bool resample = a.dev->resample != 0;
  double ll = a.dev->logLikelihood, mx = a.dev->mx, ess = a.dev->ess, lW = a.dev->lW;
  double lw = active ? a.lws[p] : 0.0;
  const double logP = log((double)a.P);

  for (int s = 0; s < a.steps; ++s) {
    // ---- resample
    int src = p;
    bool gather = resample && status == BIHIP_OK;
    if (gather) {
      const double l[1] = {lw};
      int anc[1];
      bool ok;
      if (a.resampler == BIHIP_SYSTEMATIC)
        ok = small_chain<BIHIP_SYSTEMATIC>(l, mx, a.P, a.P, a.seed, (uint32_t)k, a.batch, chain,
                                           anc);
      else if (a.resampler == BIHIP_STRATIFIED)
        ok = small_chain<BIHIP_STRATIFIED>(l, mx, a.P, a.P, a.seed, (uint32_t)k, a.batch, chain,
                                           anc);
      else
        ok = small_chain<BIHIP_MULTINOMIAL>(l, mx, a.P, a.P, a.seed, (uint32_t)k, a.batch, chain,
                                            anc);
      if (ok) {
        src = anc[0];
        if (active) a.as[p] = src;
      } else {
        status = BIHIP_DEGENERATE;
        gather = false;
      }
    }

    // ---- predict + correct
    const double t1 = a.t0 + k * a.dt, t2 = a.t0 + (k + 1) * a.dt;
    const uint32_t step = (uint32_t)(k + 1);
    double nlw = __builtin_nan("");
    if (active) {
      const T* Xin = static_cast<const T*>(a.X[s & 1]);
      T* Xout = static_cast<T*>(a.X[1 - (s & 1)]);
      T x[DL];
#pragma unroll
      for (int i = 0; i < DL; ++i) x[i] = Xin[(size_t)i * a.ld + src];
      M m(a.m);
      if constexpr (is_generated<M>::value) {
        m.template transition<INTEG, true>(grp, x, t1, t2, a.m, a.seed, a.batch, (uint32_t)p,
                                           step);
      } else {
        if constexpr (M::NOISE_FIRST) noise_first(m, a.seed, a.batch, p, step);
        if constexpr (INTEG == BIHIP_RK4) integrate_rk4(m, grp, x, t1, t2, a.m.h0);
        else integrate_dopri5(m, grp, x, t1, t2, a.m);
        if constexpr (!M::NOISE_FIRST) noise_after(m, a.seed, a.batch, p, 0, step, x);
      }
#pragma unroll
      for (int i = 0; i < DL; ++i) Xout[(size_t)i * a.ld + p] = x[i];
      const double part = obs_of(m, x, a.y + (size_t)k * a.nobs, 0, &a.m);
      nlw = (gather ? ll : lw) + part;
    }

    // ---- partials of TRANS_BLOCK particles, as block_weight_partial forms them
    double* const wm = wmax[s & 1];
    const double vm = wave_max(nlw);
    if (lane == 0) wm[w] = vm;
    __syncthreads();  // also: the new states are visible to the next step's gather
    auto max4 = [&](int q) {
      double r = wm[WPB * q];
#pragma unroll
      for (int i = 1; i < WPB; ++i) r = nan_max(r, wm[WPB * q + i]);
      return r;
    };
    const double z = nanexp(nlw - max4(w / WPB));
    const double v1 = wave_sum(z), v2 = wave_sum(z * z);
    if (lane == 0) {
      w1[w] = v1;
      w2[w] = v2;
    }
    __syncthreads();
    // ---- their combination (reduce.hip): lane quad q holds partial q, the
    // butterfly's first two exchanges add the four
    const int q = lane & (NB - 1);
    const double mq = q < nb ? max4(q) : __builtin_nan("");
    double M4 = xor_step<1>(mq, [](double x, double y) { return nan_max(x, y); });
    M4 = xor_step<2>(M4, [](double x, double y) { return nan_max(x, y); });
    double c1 = 0.0, c2 = 0.0;
    if (q < nb) {
      double b = w1[WPB * q], c = w2[WPB * q];
#pragma unroll
      for (int i = 1; i < WPB; ++i) {
        b += w1[WPB * q + i];
        c += w2[WPB * q + i];
      }
      if (b != 0.0) {
        const double f = exp(mq - M4);
        c1 = b * f;
        c2 = c * (f * f);
      }
    }
    c1 += dpp<QP_XOR1>(c1);
    c1 += dpp<QP_XOR2>(c1);
    c2 += dpp<QP_XOR1>(c2);
    c2 += dpp<QP_XOR2>(c2);

    // ---- BootstrapPF::correct's bookkeeping (pf_bookkeeping)
    ess = c1 * c1 / c2;
    lW = M4 + log(c1) - logP;
    if (p == 0) {
      a.hist.resampled[k] = gather ? 1 : 0;
      a.hist.logIncrements[k] = lW - ll;
      a.hist.ess[k] = ess;
    }
    ll = lW;
    mx = M4;
    resample = ess < a.essRel * (double)a.P;
    lw = nlw;
    ++k;
  }
  if (active) a.lws[p] = lw;
  if (p == 0) {
    a.dev->k = k;
    a.dev->status = status;
    a.dev->resample = resample ? 1 : 0;
    a.dev->logLikelihood = ll;
    a.dev->mx = mx;
    a.dev->ess = ess;
    a.dev->lW = lW;
  }
}

namespace {
// Instructions of a particle's interval: of one right-hand side and of what is not
// the integrator (variates, actions, density; generated functors count theirs).
template <class M>
void model_work(double& rhs, double& rest) {
  if constexpr (is_generated<M>::value) {
    rhs = M::RHS_WORK;
    rest = M::ONCE_WORK;
  } else {
    rhs = M::D == 2 ? 10.0 : 1.0;
    rest = 250.0;
  }
}

struct SmallFilterRunner {
  SmallFilterArgs a;
  int integ;
  hipStream_t s;
  bool only_ask;
  double d, rhs, rest;  // the answer
  template <class M>
  int run() {
    if constexpr (small_filter_model<M>()) {
      if (only_ask) {
        d = M::D;
        model_work<M>(rhs, rest);
        return BIHIP_OK;
      }
      const dim3 block(ceil_div(a.P, TRANS_BLOCK) * TRANS_BLOCK);
      if (integ == BIHIP_RK4)
        hipLaunchKernelGGL((k_filter_small<M, BIHIP_RK4>), dim3(1), block, 0, s, a);
      else
        hipLaunchKernelGGL((k_filter_small<M, BIHIP_DOPRI5>), dim3(1), block, 0, s, a);
      BIHIP_LAUNCH_CHECK();
      return BIHIP_OK;
    } else {
      return only_ask ? BIHIP_EINVAL
                      : set_error(BIHIP_EINVAL, "not a model of the one-workgroup filter");
    }
  }
};

int with_small_model(const bihip_model* m, SmallFilterRunner& r) {
  const bool f64 = m->precision == BIHIP_F64;
  if (m->model >= BIHIP_MODEL_GENERATED) return with_generated(m, r);
  if (m->model == BIHIP_MODEL_PZ) return f64 ? r.run<PZ<double>>() : r.run<PZ<float>>();
  if (m->model == BIHIP_MODEL_LG) return f64 ? r.run<LG<double>>() : r.run<LG<float>>();
  return r.only_ask ? BIHIP_EINVAL
                    : set_error(BIHIP_EINVAL, "not a model of the one-workgroup filter");
}
}  // namespace

// Instructions of one particle's interval of length dt, as far as the model and
// its settings tell: of its integrator steps and of the rest.  DOPRI5 chooses its
// steps itself; h0 is taken for its step at a tolerance of 1e-5, and the step for
// others from its order.
struct IntervalWork {
  double steps, rest;
};
static int interval_work(const bihip_model* m, double dt, IntervalWork& w) {
  SmallFilterRunner r{};
  r.only_ask = true;
  const int rc = with_small_model(m, r);
  if (rc) return rc;
  w = {0.0, r.rest};
  if (r.rhs == 0.0) return BIHIP_OK;  // no ode
  double n = m->h0 > 0.0 ? std::fmax(1.0, std::ceil(dt / m->h0 - 1e-6)) : 1e9;
  if (m->integrator == BIHIP_RK4) {
    w.steps = n * (4.0 * r.rhs + 12.0 * r.d + 12.0);
    return BIHIP_OK;
  }
  const double tol = std::fmax(1e-14, std::fmin(m->atol, m->rtol));
  n = std::fmin(n * std::fmax(1.0, std::pow(1e-5 / tol, 0.2)), (double)m->nsteps);
  w.steps = n * (7.0 * r.rhs + 34.0 * r.d + (m->precision == BIHIP_F64 ? 150.0 : 40.0));
  return BIHIP_OK;
}

// One workgroup saves launches.  It pays, above 256 particles, with w waves a SIMD
// that wait for each other, so the integrator's share of an interval is bounded,
// from predator-prey intervals of 76 instructions an RK4 step: us a step, 256 a
// call, with one workgroup and with three launches,
//   FP64 10 steps: 9.0 / 13.9 at w = 2, 12.0 / 14.7 at 3, 14.8 / 15.5 at 4;
//        50 steps: 18.9 / 20, 25.8 / 21, 32.4 / 22;
//   FP32 10 steps: 7.4 / 13.2, 9.5 / 14.2, 11.7 / 14.9;
//        100 steps: 22.7 / 30, 28.8 / 31, 36.6 / 32;
//        500 steps: 90 / 106, 115 / 106, 146 / 107.
// And each launch first fetches the whole step's code, tens of KB for a model with
// binomial draws: one step a call of SIRStochastic.bi takes 25.4 us at 500
// particles and 33 at 700, against 14.9 and 15.4 (SIR.bi 23.3 at 500 against 16.6,
// 16.5 at 100 against 15.1 but 10.1 in calls of many steps).
bool small_filter_fits(const bihip_model* m, int P, bool one_delta, double dt) {
  if (P <= 0 || P > SMALL_BLOCK) return false;
  if (m->model >= BIHIP_MODEL_GENERATED && !one_delta) return false;
  constexpr double STEPS_F64[5] = {0.0, 1e30, 5300.0, 2000.0, 1000.0};
  constexpr double STEPS_F32[5] = {0.0, 1e30, 40000.0, 10000.0, 4000.0};
  constexpr double REST[5] = {0.0, 1500.0, 700.0, 500.0, 400.0};
  const int w = ceil_div(P, TRANS_BLOCK);
  IntervalWork i;
  if (interval_work(m, dt, i) != BIHIP_OK) return false;
  return i.steps <= (m->precision == BIHIP_F64 ? STEPS_F64 : STEPS_F32)[w] && i.rest <= REST[w];
}

// A launch lasts a few milliseconds at most where the estimate of the interval
// holds (2.5 ns an instruction and wave); one step always fits.
int small_filter_steps(const bihip_model* m, double dt) {
  IntervalWork i;
  if (interval_work(m, dt, i) != BIHIP_OK) return 1;
  return (int)std::fmin(128.0, std::fmax(1.0, 1e6 / (i.steps + i.rest)));
}

int launch_small_filter(const SmallFilterLaunch& L, hipStream_t s) {
  if (L.P <= 0 || L.P > SMALL_BLOCK || L.steps < 0)
    return set_error(BIHIP_EINVAL, "the one-workgroup filter takes up to %d particles",
                     SMALL_BLOCK);
  if (L.steps == 0) return BIHIP_OK;
  SmallFilterRunner r{};
  r.a.m = to_args(L.model);
  r.a.X[0] = L.X;
  r.a.X[1] = L.Xother;
  r.a.ld = L.ld;
  r.a.P = L.P;
  r.a.steps = L.steps;
  r.a.resampler = L.resampler;
  r.a.nobs = L.nobs;
  r.a.as = L.as;
  r.a.lws = L.lws;
  r.a.dev = L.dev;
  r.a.hist = L.hist;
  r.a.y = L.y;
  r.a.t0 = L.t0;
  r.a.dt = L.dt;
  r.a.essRel = L.essRel;
  r.a.seed = L.seed;
  r.a.batch = L.batch;
  r.integ = L.model->integrator;
  r.s = s;
  return with_small_model(L.model, r);
}

}  // namespace bihip
