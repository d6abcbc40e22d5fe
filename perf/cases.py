"""Performance cases of the particle-filter library: the work that a program has it do, over
the range of sizes, models, precisions and resamplers that it is used with.

A case is one whole call sequence through the Python binding: a filter run (initial
particles, T observation intervals, the log-likelihood outputs), a bank or a batch of
filters, one step of a primitive, a training call.  Truth trajectories, observations,
particle ensembles and networks are made here from the seed (numpy and torch), so they do
not depend on the code under measurement.

`exact` restates the double-precision paths in plain torch: the Philox streams, the
integrators, the resamplers and their permuted ancestors, the networks without their
bfloat16 rounding.  The single-precision filters have no such value: one ancestor that a
rounding moves re-labels many particles, which then draw other noise.  They return their
log-likelihoods, compared within the Monte Carlo change that such re-labelling makes; their
transition is compared by itself (`transition-...`).  The double-precision filters return
their particles, weights and effective sample sizes too.
"""
import ctypes
import math

import numpy as np
import torch

from libbi_amd import capi

DAY, DT = 1.0, 0.05
SPREAD = 0.3  # of the initial particles: a filter that follows its observations has about this
RESAMPLERS = {"systematic": capi.SYSTEMATIC, "stratified": capi.STRATIFIED,
              "multinomial": capi.MULTINOMIAL}
SURROGATE_DIMS = [41, 256, 256, 256, 40]
GUIDED_DIMS = [301, 256, 256, 256, 400]


def listed():
    return [
        # the smallest filter a parameter study runs thousands of times: the user guide's
        # predator-prey model compiled from its model file; launches and latency
        {"name": "file-pz-1k", "kind": "filter", "model": "PZ.bi", "d": 2, "bits": 64, "P": 1000,
         "T": 20, "resampler": "stratified", "ess": 0.5, "graph": False},
        # the predator-prey filter of the user guide at its usual size, replayed as graphs,
        # resampling at every observation
        {"name": "pz-4k-graph", "kind": "filter", "model": "pz", "d": 2, "bits": 64, "P": 4096,
         "T": 100, "resampler": "systematic", "ess": 1.0, "graph": True},
        # the benchmark's filter: Lorenz-96 d = 40, a million particles, single-precision state
        # (its effective sample size is small, so a longer run is no longer comparable)
        {"name": "l96-1m", "kind": "filter", "model": "l96", "d": 40, "bits": 32, "P": 1 << 20,
         "T": 10, "resampler": "systematic", "ess": 0.5, "graph": False},
        # an ordinary odd size, multinomial resampling
        {"name": "l96-100k-multinomial", "kind": "filter", "model": "l96", "d": 40, "bits": 32,
         "P": 100003, "T": 8, "resampler": "multinomial", "ess": 0.5, "graph": False},
        # a double-precision filter whose particles and weights are kept
        {"name": "l96-30k-f64", "kind": "filter", "model": "l96", "d": 40, "bits": 64, "P": 30011,
         "T": 10, "resampler": "stratified", "ess": 0.5, "graph": False},
        # one interval of the simulator and the observation density, as data assimilation
        # loops and the surrogate's training data call them
        {"name": "transition-200k", "kind": "transition", "d": 40, "bits": 32, "P": 200001},
        # the inner filters of SMC^2 over the forcing, d = 200: one filter bank
        {"name": "bank-d200", "kind": "bank", "d": 200, "B": 16, "P": 16384, "T": 5,
         "net": False},
        # the inner filters of SMC^2 on the predator-prey model, uneven sizes, one batch
        {"name": "batch-pz-1024", "kind": "batch", "B": 1024, "Nmin": 256, "Nmax": 16384,
         "T": 20},
        # the learned flow in the inner filters of SMC^2 over the forcing
        {"name": "surrogate-bank", "kind": "bank", "d": 40, "B": 64, "P": 4096, "T": 8,
         "net": True},
        # the learned proposal with its weight correction, one call
        {"name": "guided-128k", "kind": "guided", "P": 1 << 17},
        # training the surrogate: one epoch of minibatches
        {"name": "train-4k", "kind": "train", "n": 1 << 16, "batch": 4096, "steps": 16},
        # the resampler's primitives one after another, as a host-driven filter calls them
        {"name": "resample-4m", "kind": "resample", "P": (1 << 22) + 13, "d": 8},
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi], odd about half of the time."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["filter", "filter", "filter", "transition", "bank", "batch", "guided",
                       "train", "resample"])
    if kind == "filter":
        model, d, bits, hi, T = rng.choice([
            ("PZ.bi", 2, 64, 1 << 18, 40), ("pz", 2, 64, 1 << 18, 100), ("pz", 2, 32, 1 << 18, 50),
            ("l96", 40, 32, 1 << 20, 8), ("l96", 40, 32, 1 << 20, 8),
            ("l96", 8, 32, 1 << 20, 16), ("l96", 200, 32, 1 << 17, 4),
            ("l96", 40, 64, 1 << 17, 8), ("Lorenz96d40.bi", 40, 32, 1 << 19, 8)])
        return {"kind": kind, "model": model, "d": d, "bits": bits,
                "P": _log_int(rng, 1000, hi), "T": rng.randint(max(2, T // 4), T),
                "resampler": rng.choice(["systematic", "stratified", "multinomial"]),
                "ess": rng.choice([0.5, 0.5, 1.0]), "graph": rng.random() < 0.4}
    if kind == "transition":
        d, bits = rng.choice([(8, 32), (40, 32), (40, 32), (200, 32), (40, 64)])
        return {"kind": kind, "d": d, "bits": bits, "P": _log_int(rng, 1000, 40 * 200001 // d)}
    if kind == "bank":
        if rng.random() < 0.5:
            return {"kind": kind, "d": 200, "B": rng.randint(2, 16),
                    "P": _log_int(rng, 1000, 16384), "T": rng.randint(2, 5), "net": False}
        return {"kind": kind, "d": 40, "B": rng.randint(2, 64), "P": _log_int(rng, 1000, 4096),
                "T": rng.randint(3, 8), "net": rng.random() < 0.6}
    if kind == "batch":
        return {"kind": kind, "B": _log_int(rng, 16, 1024), "Nmin": _log_int(rng, 64, 512),
                "Nmax": _log_int(rng, 1024, 16384), "T": rng.randint(5, 20)}
    if kind == "guided":
        return {"kind": kind, "P": _log_int(rng, 1000, 1 << 17)}
    if kind == "train":
        return {"kind": kind, "n": _log_int(rng, 1 << 13, 1 << 16),
                "batch": 64 * rng.randint(16, 64), "steps": rng.randint(4, 16)}
    return {"kind": kind, "P": _log_int(rng, 1000, 1 << 22), "d": rng.randint(2, 8)}


# ---------------------------------------------------------------- synthetic data
def _l96_rhs(x, F):
    m = np if isinstance(x, np.ndarray) else torch
    if m is np:
        return (np.roll(x, -1, 0) - np.roll(x, 2, 0)) * np.roll(x, 1, 0) - x + F
    return (torch.roll(x, -1, 0) - torch.roll(x, 2, 0)) * torch.roll(x, 1, 0) - x + F


def _rk4(f, x, h):
    a = f(x)
    b = f(x + 0.5 * h * a)
    c = f(x + 0.5 * h * b)
    return x + h / 6.0 * (a + 2.0 * b + 2.0 * c + f(x + h * c))


def _l96_truth(rng, d, T, F=8.0, flow=None):
    """A point on the attractor and T observations of the even dimensions, every 0.05."""
    x = F + 0.5 * rng.standard_normal(d)
    for _ in range(300):
        x = _rk4(lambda u: _l96_rhs(u, F), x, 0.025)
    x0, y = x.copy(), np.empty((T, d // 2))
    for k in range(T):
        if flow is not None:
            x = flow(x)
        else:
            for _ in range(2):
                x = _rk4(lambda u: _l96_rhs(u, F), x, DT / 2)
        x = x + 0.1 * rng.standard_normal(d)
        y[k] = x[0::2] + rng.standard_normal(d // 2)
    return x0, y


def _pz_rhs(x, alpha, c=0.25, e=0.3, ml=0.1, mq=0.1):
    P, Z = x[0], x[1]
    k = (alpha * P - c * P * Z, e * c * P * Z - ml * Z - mq * Z * Z)
    return np.array(k) if isinstance(x, np.ndarray) else torch.stack(k)


def _pz_truth(rng, T):
    x, y = np.array([2.0, 2.0]), np.empty((T, 1))
    for k in range(T):
        alpha = 0.5 + 0.2 * rng.standard_normal()
        for _ in range(10):
            x = _rk4(lambda u: _pz_rhs(u, alpha), x, 0.1)
        y[k, 0] = math.exp(math.log(x[0]) + 0.2 * rng.standard_normal())
    return y


def _l96_ensemble(rng, seed, d, P, dtype):
    """P states around a trajectory on the attractor, as a filter's particles lie (d x P)."""
    x0, y = _l96_truth(rng, d, 1)
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((d, P), generator=g, device="cuda", dtype=torch.float32)
    x = torch.from_numpy(x0).to("cuda", torch.float32)[:, None] + 0.7 * x
    return _rk4(lambda u: _l96_rhs(u, 8.0), x, DT / 2).to(dtype).contiguous(), y


def _network(rng, dims, gain=1.2):
    """Weights and biases of a network with activations of order one."""
    return [((gain / math.sqrt(m)) * rng.standard_normal((n, m))).astype(np.float32)
            if k == 0 else (0.05 * rng.standard_normal(n)).astype(np.float32)
            for m, n in zip(dims[:-1], dims[1:]) for k in (0, 1)]


def _forward(net, u, one=np):
    """The network in the precision of u (last axis: features)."""
    L = len(net) // 2
    for k in range(L):
        u = u @ net[2 * k].T + net[2 * k + 1]
        if k + 1 < L:
            u = u / (1.0 + one.exp(-1.702 * u))
    return u


def _mlp(ctx, dims, net):
    m = capi.MLP(ctx, dims, seed=1)
    m.set_params(np.concatenate([p.reshape(-1) for p in net]))
    return m


def _population(case, rng):
    """SMC^2's population: sizes log-uniform, theta = (mu, sigma, c, e) from log-normals."""
    B = case["B"]
    N = np.floor(np.exp(rng.uniform(np.log(case["Nmin"]), np.log(case["Nmax"]), B)))
    th = [np.exp(rng.normal(np.log(m), s, B))
          for m, s in ((0.5, 0.2), (0.2, 0.2), (0.25, 0.1), (0.3, 0.1))]
    return N.astype(np.int32), np.stack(th, axis=1)


def _data(case, seed):
    """The seed's inputs on the host, shared by prepare and exact."""
    rng = np.random.default_rng(seed)
    s = {"seed": seed & 0x7FFFFFFF}
    kind = case["kind"]
    if kind == "filter":
        if case["d"] == 2:
            s["y"], s["x0"] = _pz_truth(rng, case["T"]), None
        else:
            s["x0"], s["y"] = _l96_truth(rng, case["d"], case["T"])
    elif kind == "bank":
        s["theta"] = np.sort(rng.uniform(7.5, 8.5, case["B"]))
        if case["net"]:
            s["net"] = _network(rng, SURROGATE_DIMS)
            net = [p.astype(np.float64) for p in s["net"]]
            s["x0"], s["y"] = _l96_truth(
                rng, case["d"], case["T"],
                flow=lambda x: x + 0.3 * _forward(net, np.append((x - 2.3) / 3.6, 0.0)))
        else:
            s["x0"], s["y"] = _l96_truth(rng, case["d"], case["T"])
    elif kind == "batch":
        s["N"], s["theta"] = _population(case, rng)
        s["y"] = _pz_truth(rng, case["T"])
    elif kind == "transition":
        dt = torch.float32 if case["bits"] == 32 else torch.float64
        s["X"], s["y"] = _l96_ensemble(rng, seed, case["d"], case["P"], dt)
    elif kind == "guided":
        s["net"] = _network(rng, GUIDED_DIMS, 0.8)
        s["X"], s["y"] = _l96_ensemble(rng, seed, 200, case["P"], torch.float32)
    elif kind == "train":
        s["net"] = _network(rng, SURROGATE_DIMS)
        g = torch.Generator(device="cuda").manual_seed(seed)
        x = torch.randn((case["n"], 41), generator=g, device="cuda")
        s["X"] = x
        s["Y"] = (torch.roll(x, -1, 1)[:, :40] - torch.roll(x, 2, 1)[:, :40]) * x[:, :40] * 0.5
    else:
        g = torch.Generator(device="cuda").manual_seed(seed)
        # log-weights of an effective sample size of about 0.3
        s["lws"] = 1.1 * torch.randn(case["P"], generator=g, device="cuda", dtype=torch.float64)
        s["X"] = torch.randn((case["d"], case["P"]), generator=g, device="cuda")
        s["a"] = float(rng.uniform())
    return s


# ---------------------------------------------------------------- the cases
def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    s = _data(case, seed)
    ctx = s["ctx"] = capi.Context(0)
    s["case"], kind = case, case["kind"]
    prec = capi.F32 if case.get("bits", 32) == 32 else capi.F64
    if kind == "filter":
        if case["model"] == "PZ.bi":
            m = capi.generated_model("PZ", precision=prec, mu=0.5, sigma=0.2)
        elif case["model"] == "Lorenz96d40.bi":
            m = capi.generated_model("Lorenz96d40", precision=prec, F=8.0, noise_sd=0.1,
                                     obs_sd=1.0, init_sd=SPREAD)
        elif case["model"] == "pz":
            m = capi.make_model("pz", precision=prec)
        else:
            m = capi.make_model("l96", d=case["d"], precision=prec, init_sd=SPREAD)
        s["f"] = capi.ParticleFilter(ctx, m, case["P"], case["T"], DAY if case["d"] == 2 else DT,
                                     s["seed"], RESAMPLERS[case["resampler"]], case["ess"],
                                     use_graph=case["graph"])
        s["f"].set_observations(s["y"])
    elif kind == "bank":
        m = capi.make_model("l96", d=case["d"], precision=capi.F32, init_sd=SPREAD)
        s["f"] = capi.FilterBank(ctx, m, case["P"], case["T"], DT, s["seed"], s["theta"],
                                 ess_rel=0.5, use_graph=True)
        if case["net"]:
            s["mlp"] = _mlp(ctx, SURROGATE_DIMS, s["net"])
            s["norm"] = capi.SurrogateNorm(x_shift=2.3, x_scale=3.6, par_shift=8.0, par_scale=1.0,
                                           dx_scale=0.3)
            s["f"].set_surrogate(s["mlp"], s["norm"])
        s["f"].set_observations(s["y"])
    elif kind == "batch":
        s["f"] = capi.BatchFilter(ctx, capi.make_model("pz", precision=capi.F64), s["N"],
                                  s["theta"], case["T"], DAY, s["seed"], ess_rel=0.5)
        s["f"].set_observations(s["y"])
    elif kind == "transition":
        s["m"] = capi.make_model("l96", d=case["d"], precision=prec)
        s["yd"] = torch.from_numpy(s["y"][0]).cuda()
    elif kind == "guided":
        s["mlp"] = _mlp(ctx, GUIDED_DIMS, s["net"])
        s["norm"] = capi.GuidedNorm(x_shift=2.3, x_scale=3.6, innov_scale=1.0, par_shift=8.0,
                                    par_scale=1.0)
    elif kind == "train":
        s["mlp"] = _mlp(ctx, SURROGATE_DIMS, s["net"])
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "filter":
        f = s["f"]
        f.init(s["x0"])
        f.step(case["T"])
        out = f.outputs()
        if case["bits"] == 32:
            return {k: out[k] for k in ("logLikelihood", "logIncrements")}
        X, _, out["lws"] = f.state()
        out["X"] = X[:, :case["P"]]
        return out
    if kind == "bank":
        s["f"].init(s["x0"])
        s["f"].step(case["T"])
        out = s["f"].outputs()
        return {k: out[k] for k in ("logLikelihood", "logIncrements")}
    if kind == "batch":
        s["f"].init()
        s["f"].step(case["T"])
        return s["f"].outputs()
    if kind == "transition":
        P, h, L = case["P"], s["ctx"].h, capi.lib()
        out = torch.empty_like(s["X"])
        n = torch.empty(P, dtype=torch.int32, device="cuda")
        lws = torch.zeros(P, dtype=torch.float64, device="cuda")
        capi.check(L.bihip_transition(h, ctypes.byref(s["m"]), s["seed"], 0, 1, 0.0, DT, P,
                                      _ptr(s["X"]), _ptr(out), P, None, _ptr(n)))
        capi.check(L.bihip_obs_logdensity(h, ctypes.byref(s["m"]), _ptr(s["yd"]), P, _ptr(out), P,
                                          _ptr(lws)))
        return {"X": out, "steps": n, "lws": lws}
    if kind == "guided":
        X = s["X"].clone()
        inc = s["mlp"].guided_propose(s["norm"], 8.0, X, s["y"][0], s["seed"], 1)
        return {"X": X, "inc": inc}
    if kind == "train":
        losses = s["mlp"].train(s["X"], s["Y"], case["batch"], case["steps"], 1e-4,
                                seed=s["seed"])
        return {"losses": losses, "params": s["mlp"].get_params()}
    P, h, L = case["P"], s["ctx"].h, capi.lib()
    X = s["X"].clone()
    Ws = torch.empty(P, dtype=torch.float64, device="cuda")
    Os, anc = (torch.empty(P, dtype=torch.int32, device="cuda") for _ in range(2))
    capi.check(L.bihip_sumexpu_inclusive_scan(h, _ptr(s["lws"]), P, _ptr(Ws), None))
    capi.check(L.bihip_systematic_cumulative_offspring(h, _ptr(Ws), P, P, s["a"], _ptr(Os)))
    capi.check(L.bihip_cumulative_offspring_to_ancestors_permute(h, _ptr(Os), P, _ptr(anc)))
    capi.check(L.bihip_gather_rows(h, _ptr(anc), P, case["d"], _ptr(X), P, 4))
    return {"Ws": Ws, "as": anc, "X": X}


def work(case):
    """Bytes: the state read and written once per interval, the log-weights read and written,
    and on resampling (every interval) the ancestors written and read.  Flops: about 3 DOPRI5
    steps of 7 stages per interval for Lorenz-96 (a right-hand side and the stage sums, 140
    per dimension and step), 10 RK4 steps for the predator-prey model."""
    kind = case["kind"]
    if kind in ("filter", "bank"):
        n = case["P"] * case["T"] * case.get("B", 1)
        d, b = case["d"], case.get("bits", 32) // 8
        fl = 1000 if d == 2 else 420 * d
        if case.get("net"):
            fl = 2 * sum(i * o for i, o in zip(SURROGATE_DIMS[:-1], SURROGATE_DIMS[1:]))
        return {"bytes": n * (2 * d * b + 24), "flops": n * fl}
    if kind == "batch":
        mean = (case["Nmax"] - case["Nmin"]) / math.log(case["Nmax"] / case["Nmin"])
        n = case["B"] * mean * case["T"]
        return {"bytes": n * 56, "flops": n * 1000}
    if kind == "transition":
        return {"bytes": case["P"] * (2 * case["d"] * case["bits"] // 8 + 12),
                "flops": case["P"] * 420 * case["d"]}
    if kind == "guided":
        return {"bytes": case["P"] * (2 * 200 * 4 + 8),
                "flops": case["P"] * 2 * sum(i * o for i, o in zip(GUIDED_DIMS[:-1],
                                                                   GUIDED_DIMS[1:]))}
    if kind == "train":
        n = case["batch"] * case["steps"]
        return {"bytes": n * 4 * 81,
                "flops": n * 6 * sum(i * o for i, o in zip(SURROGATE_DIMS[:-1],
                                                           SURROGATE_DIMS[1:]))}
    return {"bytes": case["P"] * (8 + 8 + 4 + 8 * case["d"]), "flops": 20 * case["P"]}


def tolerance(case):
    """About four times what another order of the same single-precision sums changes (stage
    sums with the forcing inside the right-hand side, activations by another exponential);
    the double-precision paths are held to what the integer weight sums and the reductions
    leave open."""
    kind = case["kind"]
    if kind == "filter" and case["bits"] == 64 or kind == "batch":
        return {"rel": 1e-10, "max": 1e-8, "differ": 1e-4}
    if kind in ("filter", "bank"):  # seen: 0.0075 over 40 cases
        return {"rel": 2e-2, "max": 0.2}
    if kind == "transition":  # seen: 9e-8, 2e-6 to 4e-6, 1.5e-4
        return {"rel": 4e-7, "max": 2e-5, "differ": 6e-4} if case["bits"] == 32 else \
            {"rel": 1e-14, "max": 1e-12, "differ": 1e-4}
    if kind == "guided":  # seen: 4e-7, 5e-5
        return {"rel": 2e-6, "max": 2e-4}
    if kind == "train":  # seen: 9e-6, 6e-4
        return {"rel": 4e-5, "max": 3e-3}
    return {"rel": 1e-12, "max": 1e-11, "differ": 1e-6}


# ---------------------------------------------------------------- 64-bit restatement
def _philox(c0, c1, c2, c3, seed):
    """Philox4x32-10 on int64 tensors of 32-bit words."""
    mask = 0xFFFFFFFF
    k0, k1 = seed & mask, (seed >> 32) & mask

    def mul(m, x):  # the product's 64 bits, wrapped into int64
        p = x * m
        return (p >> 32) & mask, p & mask

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c0)
        h1, l1 = mul(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return c0, c1, c2, c3


def _words(p, step, tag, batch, block, seed):
    z = torch.zeros_like(p)
    return _philox(p, z + step, z + (tag | (batch << 8)), z + block, seed)


def _pairs(r0, r1, bits):
    if bits == 32:  # the top 24 bits of each word
        u1, u2 = 1.0 - (r0 >> 8).double() * 2.0**-24, (r1 >> 8).double() * 2.0**-24
    else:
        u1, u2 = 1.0 - r0.double() * 2.0**-32, r1.double() * 2.0**-32
    rad = torch.sqrt(-2.0 * torch.log(u1))
    return rad * torch.cos(2.0 * math.pi * u2), rad * torch.sin(2.0 * math.pi * u2)


def _normals(p, step, tag, batch, n, seed, bits):
    """n normals per particle (n x ...): normal j from block j / 4."""
    z = []
    for b in range((n + 3) // 4):
        r = _words(p, step, tag, batch, b, seed)
        z += [*_pairs(r[0], r[1], bits), *_pairs(r[2], r[3], bits)]
    return torch.stack(z[:n])


def _u53(p, step, tag, batch, seed):
    r = _words(p, step, tag, batch, 0, seed)
    return ((r[0] << 21) | (r[1] >> 11)).double() * 2.0**-53


A = [[], [0.2], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
     [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
     [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656],
     [35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]]
ERR = [71 / 57600, 0.0, -71 / 16695, 71 / 1920, -17253 / 339200, 22 / 525, -1 / 40]


def _dopri5(f, x, t, t2, h0=0.05, tol=1e-5):
    """Adaptive DOPRI5 of every particle (columns of x) with its own step: x and the steps."""
    h = torch.full(x.shape[1:], h0, dtype=x.dtype, device=x.device)
    t = torch.full_like(h, t)
    old = torch.full_like(h, math.log(1e-4))
    n = torch.zeros_like(h, dtype=torch.int32)
    k1 = f(x)
    while bool((t < t2).any()):
        on = t < t2
        h = torch.where(t + 1.01 * h - t2 > 0.0, t2 - t, h)
        k = [k1]
        for s in range(1, 7):
            xs = x + h * sum(a * q for a, q in zip(A[s], k) if a != 0.0)
            k.append(f(xs))
        e = h * sum(a * q for a, q in zip(ERR, k) if a != 0.0)
        e = e / (tol + tol * torch.maximum(x.abs(), xs.abs()))
        e2 = (e * e).mean(0)
        ok = on & (e2 <= 1.0)
        t = torch.where(ok, t + h, t)
        x, k1 = torch.where(ok, xs, x), torch.where(ok, k[6], k1)
        lf = 0.5 * (0.2 - 0.04 * 0.75) * torch.log(e2)
        up = torch.clamp(torch.exp(0.04 * old + math.log(0.9) - lf), 0.2, 10.0)
        down = torch.clamp(torch.exp(math.log(0.9) - lf), min=0.2)
        h = torch.where(on, h * torch.where(ok, up, down), h)
        old = torch.where(ok, 0.5 * torch.log(torch.clamp(e2, min=1e-8)), old)
        n += on.int()
    return x, n


def _ancestors(lws, N, k, batch, seed, resampler):
    """Permuted ancestors of every row (filters of N_r particles, padded with -inf)."""
    idx = torch.arange(lws.shape[1], device=lws.device)[None, :]
    live = idx < N
    w = torch.exp(lws - lws.amax(1, keepdim=True))
    Ws = torch.cumsum(w, 1)
    r = Ws / Ws[:, -1:] * N
    if resampler == "systematic":
        o = r + _u53(torch.zeros_like(batch), k, capi.TAG_SYSTEMATIC, batch, seed)
    else:
        c = torch.minimum(r.long(), N - 1)
        o = r + _u53(c, k, capi.TAG_STRATIFIED, batch, seed)
    O = torch.minimum(o.long(), N)
    o = torch.diff(O, dim=1, prepend=torch.zeros_like(O[:, :1]))
    e, fr = torch.clamp(o - 1, min=0), ((o == 0) & live).long()
    E, Fk = torch.cumsum(e, 1) - e, torch.cumsum(fr, 1) - fr
    own = torch.searchsorted(E.contiguous(), Fk.contiguous(), right=True) - 1
    return torch.where((fr == 0), idx.expand_as(own), own)


def _exact_filters(model, y, N, theta, T, seed, resampler, ess_rel, x0, d):
    """Rows of double-precision bootstrap filters: state (d x R x P), log-weights, outputs."""
    R, P = len(N), int(max(N))
    dev = "cuda"
    N = torch.as_tensor(np.asarray(N, np.int64), device=dev)[:, None]
    th = torch.as_tensor(theta, dtype=torch.float64, device=dev)
    batch = torch.arange(R, device=dev)[:, None]
    p = torch.arange(P, device=dev)[None, :].expand(R, P)
    live = p < N
    z = _normals(p, 0, capi.TAG_INIT, batch, d, seed, 64)
    if model == "pz":
        x = torch.stack([torch.exp(math.log(2.0) + 0.2 * z[0]), torch.exp(math.log(2.0) + 0.1 * z[1])])
    else:
        x = torch.as_tensor(x0, device=dev)[:, None, None] + SPREAD * z
    ll = torch.zeros((R, 1), dtype=torch.float64, device=dev)
    lws = torch.where(live, 0.0, -math.inf).double()
    res = torch.zeros((R, 1), dtype=torch.bool, device=dev)
    li, es, rs = [], [], []
    y = torch.as_tensor(y, device=dev)
    for k in range(T):
        if bool(res.any()):
            a = _ancestors(lws, N, k, batch, seed, resampler)
            a = torch.where(res, a, p)
            x = torch.gather(x, 2, a[None].expand_as(x))
            lws = torch.where(live & res, ll, lws)
        rs.append(res)
        if model == "pz":
            z = _normals(p, k + 1, capi.TAG_NOISE, batch, 1, seed, 64)[0]
            mu, sg, c, e = (th[:, i:i + 1] for i in range(4))
            al = mu + sg * z
            for _ in range(10):
                x = _rk4(lambda u: _pz_rhs(u, al, c, e), x, 0.1)
            r = (torch.log(y[k, 0]) - torch.log(x[0])) / 0.2
            ob = -0.5 * r * r - 0.5 * math.log(2 * math.pi) - torch.log(0.2 * y[k, 0])
        else:
            x, _ = _dopri5(lambda u: _l96_rhs(u, 8.0), x, k * DT, (k + 1) * DT)
            x = x + 0.1 * _normals(p, k + 1, capi.TAG_NOISE, batch, d, seed, 64)
            r = y[k][:, None, None] - x[0::2]
            ob = (-0.5 * r * r - 0.5 * math.log(2 * math.pi)).sum(0)
        lws = torch.where(live, lws + ob, -math.inf)
        mx = lws.amax(1, keepdim=True)
        w = torch.exp(lws - mx)
        s1, s2 = w.sum(1, keepdim=True), (w * w).sum(1, keepdim=True)
        lW = mx + torch.log(s1) - torch.log(N.double())
        li.append(lW - ll)
        es.append(s1 * s1 / s2)
        ll = lW
        res = es[-1] < ess_rel * N.double()
    row = lambda v: torch.cat(v, 1)  # noqa: E731
    return x, lws, {"logLikelihood": ll[:, 0], "logIncrements": row(li), "ess": row(es)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "bank" or kind == "filter" and case["bits"] == 32:
        return None
    if kind == "filter" and (case["resampler"] == "multinomial" or
                             case["P"] * case["T"] * case["d"] > 2e8):
        return None
    s = _data(case, seed)
    if kind in ("filter", "batch"):
        one = kind == "filter"
        x, lws, out = _exact_filters(
            "pz" if one is False or case["d"] == 2 else "l96", s["y"],
            [case["P"]] if one else s["N"], [[0.5, 0.2, 0.25, 0.3]] if one else s["theta"],
            case["T"], s["seed"], case["resampler"] if one else "systematic",
            case["ess"] if one else 0.5, s.get("x0"), case.get("d", 2))
        out["resampled"] = None
        if one:
            out["logIncrements"], out["ess"] = out["logIncrements"][0], out["ess"][0]
            out["logLikelihood"] = float(out["logLikelihood"][0])
            out["lws"], out["X"] = lws[0], x[:, 0]
        else:
            out["status"] = None
        return out
    if kind == "transition":
        x, _ = _dopri5(lambda u: _l96_rhs(u, 8.0), s["X"].double(), 0.0, DT)
        p = torch.arange(case["P"], device="cuda")
        x = x + 0.1 * _normals(p, 1, capi.TAG_NOISE, 0, case["d"], s["seed"], case["bits"])
        r = torch.from_numpy(s["y"][0]).cuda()[:, None] - x[0::2]
        return {"X": x, "steps": None,
                "lws": (-0.5 * r * r - 0.5 * math.log(2 * math.pi)).sum(0)}
    if kind == "guided":
        net = [torch.from_numpy(w).cuda().double() for w in s["net"]]
        X, y = s["X"].double(), torch.from_numpy(s["y"][0]).cuda()[:, None]
        u = torch.cat([(X - 2.3) / 3.6, y - X[0::2], torch.zeros_like(X[:1])])
        o = _forward(net, u.T, torch).T
        m, v = o[:200], o[200:]
        z = _normals(torch.arange(case["P"], device="cuda"), 1, capi.TAG_NOISE, 0, 200, s["seed"],
                     32)
        q = m + torch.exp(0.5 * v) * z
        X = X + 0.1 * q
        r = y - X[0::2]
        inc = (-0.5 * q * q + 0.5 * z * z + 0.5 * v).sum(0)
        return {"X": X, "inc": inc + (-0.5 * r * r - 0.5 * math.log(2 * math.pi)).sum(0)}
    if kind == "train":
        return _exact_train(case, s)
    w = torch.exp(s["lws"] - s["lws"].max())
    return {"Ws": torch.cumsum(w, 0), "as": None, "X": None}


def _exact_train(case, s):
    """The minibatches of the keyed shuffle and Adam on the network in 64 bits."""
    n, batch, seed = case["n"], case["batch"], s["seed"]
    net = [torch.from_numpy(w).double().cuda().requires_grad_() for w in s["net"]]
    X, Y = s["X"].double(), s["Y"].double()
    m1, m2 = [torch.zeros_like(w) for w in net], [torch.zeros_like(w) for w in net]
    perm, pos, epoch, losses = list(range(n)), n, -1, []
    at = torch.arange(n)
    for it in range(case["steps"]):
        if pos + batch > n:
            epoch, pos = epoch + 1, 0
            u = _u53(at, epoch, 12, 0, seed)  # 12: the minibatch shuffle's stream
            j = torch.minimum(at, (u * (at + 1).double()).long()).tolist()
            for i in range(n - 1, 0, -1):
                perm[i], perm[j[i]] = perm[j[i]], perm[i]
        idx = torch.tensor(perm[pos:pos + batch], device="cuda")
        pos += batch
        loss = (_forward(net, X[idx], torch) - Y[idx]).square().mean()
        losses.append(loss.detach())
        g = torch.autograd.grad(loss, net)
        b1, b2 = 1.0 - 0.9**(it + 1), 1.0 - 0.999**(it + 1)
        with torch.no_grad():
            for w, q, a, b in zip(net, g, m1, m2):
                a.mul_(0.9).add_(0.1 * q)
                b.mul_(0.999).add_(0.001 * q * q)
                w -= 1e-4 * (a / b1) / ((b / b2).sqrt() + 1e-8)
    return {"losses": torch.stack(losses), "params": torch.cat([w.detach().reshape(-1) for w in net])}
