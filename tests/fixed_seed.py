"""Outputs of fixed calls as CRC-32 of their bytes (tests/golden/fixed_seed_results.json,
test_gpu_fixed_seed.py).  A filter's particles follow from the last bits of its
single-precision arithmetic: one ancestor that moves relabels the particles after it,
which then draw other noise.  So a change that only regroups the arithmetic of a kernel
shows here and nowhere else.

Written by `python tests/fixed_seed.py`, on an MI355X; only where a change of the results
is meant.
"""
import ctypes
import json
import os
import sys
import zlib

import numpy as np

if __name__ == "__main__":
    sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from libbi_amd import capi, guided, surrogate

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden",
                      "fixed_seed_results.json")


def l96_state(d):
    """A point near the Lorenz-96 attractor, from elementary float64 operations only."""
    x = 8.0 + 0.01 * np.arange(d) * (-1.0) ** np.arange(d)

    def f(u):
        return (np.roll(u, -1) - np.roll(u, 2)) * np.roll(u, 1) - u + 8.0
    for _ in range(400):
        a = f(x)
        b = f(x + 0.0125 * a)
        c = f(x + 0.0125 * b)
        x = x + 0.025 / 6.0 * (a + 2.0 * b + 2.0 * c + f(x + 0.025 * c))
    return np.ascontiguousarray(x)


def observations(d, T):
    y = l96_state(d)[0::2][None, :] + 0.8 * np.random.default_rng(d).standard_normal((T, d // 2))
    return np.ascontiguousarray(y)


def crc(*arrays):
    c = 0
    for a in arrays:
        c = zlib.crc32(np.ascontiguousarray(a).tobytes(), c)
    return c


def _transition(ctx, torch, d, prec, integ, quirk, P):
    """Initial particles, one interval, its flow and the observation density."""
    L = capi.lib()
    # several steps in an interval, some rejected
    m = capi.make_model("l96", d=d, precision=prec, integrator=integ, h0=0.02, atol=1e-6,
                        rtol=1e-6)
    m.host_quirk = quirk
    dt = torch.float64 if prec == capi.F64 else torch.float32
    X = torch.empty((d, P), dtype=dt, device="cuda")
    Y = torch.empty_like(X)
    lws = torch.zeros(P, dtype=torch.float64, device="cuda")
    y = torch.from_numpy(observations(d, 1)[0]).cuda()
    mean = l96_state(d)
    torch.cuda.synchronize()
    capi.check(L.bihip_init_samples(ctx.h, ctypes.byref(m), 21, 0, P, capi.ptr(X), P,
                                    mean.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
    capi.check(L.bihip_transition(ctx.h, ctypes.byref(m), 5, 0, 1, 0.0, 0.05, P, capi.ptr(X),
                                  capi.ptr(Y), P, None, None))
    capi.check(L.bihip_obs_logdensity(ctx.h, ctypes.byref(m), capi.ptr(y), P, capi.ptr(Y), P,
                                      capi.ptr(lws)))
    ctx.sync()
    out = [X.cpu().numpy(), Y.cpu().numpy(), lws.cpu().numpy()]
    capi.check(L.bihip_flow(ctx.h, ctypes.byref(m), 0.05, 0.1, P, capi.ptr(Y), P, None, None))
    ctx.sync()
    return crc(*out, Y.cpu().numpy())


def _filter(ctx, model, d, P, T, resampler=capi.SYSTEMATIC, learn=None):
    """States, log-weights, log-likelihood increments and effective sample sizes after T
    intervals."""
    f = capi.ParticleFilter(ctx, model, P, T, 0.05, 7, resampler, 0.5)
    f.set_observations(observations(d, T))
    if learn is not None:
        learn(f)
    f.init(l96_state(d))
    f.step(T)
    out = f.outputs()
    X, _, lws = f.state()
    r = crc(X[:, :P].cpu().numpy(), lws.cpu().numpy(), out["logIncrements"], out["ess"])
    f.close()
    return r


def _bank(ctx, d, B, P, T, learn=None):
    """Increments, effective sample sizes and the last filter's states of a bank."""
    m = capi.make_model("l96", d=d, precision=capi.F32, init_sd=0.3)
    b = capi.FilterBank(ctx, m, P, T, 0.05, 11, np.linspace(7.6, 8.4, B), ess_rel=0.5)
    if learn is not None:
        learn(b)
    b.set_observations(observations(d, T))
    b.init(l96_state(d))
    b.step(T)
    out = b.outputs()
    X = b.state(B - 1)[0]
    r = crc(out["logIncrements"], out["ess"], X[:, :P].cpu().numpy())
    b.close()
    return r


SURROGATE_NORM = capi.SurrogateNorm(x_shift=2.3, x_scale=3.6, par_shift=8.0, par_scale=1.0,
                                    dx_scale=0.3)
GUIDED_NORM = capi.GuidedNorm(x_shift=2.3, x_scale=3.6, innov_scale=1.0, par_shift=8.0,
                              par_scale=1.0)


def _states(torch, d, P):
    x = 2.3 + 3.6 * np.random.default_rng(P).standard_normal((d, P))
    x = torch.from_numpy(x.astype(np.float32)).cuda()
    torch.cuda.synchronize()
    return x


def _surrogate_flow(ctx, torch):
    net = capi.MLP(ctx, surrogate.DIMS, seed=4)
    out = net.surrogate_flow(SURROGATE_NORM, 8.1, _states(torch, 40, 3001))
    ctx.sync()
    r = crc(out.cpu().numpy())
    net.close()
    return r


def _guided_propose(ctx, torch):
    net = capi.MLP(ctx, guided.DIMS, seed=5)
    X = _states(torch, 200, 3001)
    inc = net.guided_propose(GUIDED_NORM, 8.2, X, observations(200, 1)[0], 5, 2)
    ctx.sync()
    r = crc(X.cpu().numpy(), inc.cpu().numpy())
    net.close()
    return r


def _learned(ctx, kind, run):
    """run(set): a filter or bank that the function `set` gives the network to."""
    surr = kind == "surrogate"
    net = capi.MLP(ctx, surrogate.DIMS if surr else guided.DIMS, seed=4)
    r = run(lambda f: f.set_surrogate(net, SURROGATE_NORM) if surr else
            f.set_guided(net, GUIDED_NORM))
    net.close()
    return r


def _training(ctx, torch, dims, n, batch, loss):
    """Gradient, minibatch losses and parameters of a short training."""
    net = capi.MLP(ctx, dims, seed=5)
    net.set_loss(loss)
    rng = np.random.default_rng(n)
    X = torch.from_numpy(rng.standard_normal((n, dims[0])).astype(np.float32)).cuda()
    m = dims[-1] // 2 if loss == capi.LOSS_GAUSS else dims[-1]
    T = torch.from_numpy(rng.standard_normal((n, m)).astype(np.float32)).cuda()
    torch.cuda.synchronize()
    _, g = net.loss_grad(X, T)
    losses = net.train(X, T, batch, 30, 1e-3, seed=3)
    r = crc(g, losses, net.get_params())
    net.close()
    return r


def cases():
    """name -> function of (context, torch)"""
    out = {}
    for d in (8, 40, 200):
        for p, prec in (("f32", capi.F32), ("f64", capi.F64)):
            for i, integ, quirk in (("dopri5", capi.DOPRI5, 0), ("host-dopri5", capi.DOPRI5, 1),
                                    ("rk4", capi.RK4, 0)):
                # d = 200: both layouts of its lanes
                for P in (5003,) if d < 200 else (
                        (5003, 66001) if (p, i) == ("f64", "rk4") else (5003, 9001)):
                    out[f"transition-l96-{d}-{p}-{i}" + (f"-{P}" if P != 5003 else "")] = (
                        lambda ctx, torch, a=(d, prec, integ, quirk, P): _transition(
                            ctx, torch, *a))
            for r, res in (("systematic", capi.SYSTEMATIC), ("multinomial", capi.MULTINOMIAL)):
                out[f"filter-l96-{d}-{p}-{r}"] = (
                    lambda ctx, torch, a=(d, prec, res): _filter(
                        ctx, capi.make_model("l96", d=a[0], precision=a[1], init_sd=0.3), a[0],
                        30011 if a[0] < 200 else 5003, 6, a[2]))
            if d == 200:
                for P in (9001,):
                    out[f"filter-l96-200-{p}-{P}"] = (
                        lambda ctx, torch, prec=prec, P=P: _filter(
                            ctx, capi.make_model("l96", d=200, precision=prec, init_sd=0.3), 200,
                            P, 4))
        out[f"bank-l96-{d}"] = lambda ctx, torch, d=d: _bank(ctx, d, 3, 2049, 5)
    out["bank-l96-200-12k"] = lambda ctx, torch: _bank(ctx, 200, 4, 3001, 4)
    out["surrogate-flow"] = _surrogate_flow
    out["guided-propose"] = _guided_propose
    for kind, d in (("surrogate", 40), ("guided", 200)):
        m = capi.make_model("l96", d=d, precision=capi.F32, init_sd=0.3)
        out[f"filter-{kind}"] = lambda ctx, torch, k=kind, m=m, d=d: _learned(
            ctx, k, lambda give: _filter(ctx, m, d, 5003, 5, learn=give))
        out[f"bank-{kind}"] = lambda ctx, torch, k=kind, d=d: _learned(
            ctx, k, lambda give: _bank(ctx, d, 3, 2049, 4, learn=give))
    for dims, n, batch in (([41, 256, 256, 256, 40], 1000, 320), ([5, 64, 3], 64, 64),
                           ([7, 65, 130, 9], 700, 64)):
        out["training-" + "-".join(map(str, dims))] = (
            lambda ctx, torch, a=(dims, n, batch): _training(ctx, torch, *a, capi.LOSS_MSE))
    out["training-gauss"] = (lambda ctx, torch: _training(ctx, torch, [20, 128, 16], 500, 128,
                                                          capi.LOSS_GAUSS))
    return out


if __name__ == "__main__":
    import torch
    ctx = capi.Context(0)
    got = {name: f(ctx, torch) for name, f in cases().items()}
    with open(GOLDEN, "w") as f:
        json.dump(got, f, indent=1, sort_keys=True)
        f.write("\n")
