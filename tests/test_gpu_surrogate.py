"""The fused surrogate flow (bihip_surrogate_flow) and the filter step that
uses it (bihip_pf_set_surrogate): the fused kernel against the GEMM path and
the oracle's MLP, the filter step against its composition (flow, Philox
noise, observation density), and a trained surrogate against the exact
integrator."""
import ctypes

import numpy as np
import pytest

from libbi_amd import capi, guided, surrogate

pytestmark = pytest.mark.gpu

D = 40


def _norm():
    return capi.SurrogateNorm(x_shift=2.3, x_scale=3.6, par_shift=8.0, par_scale=1.0,
                              dx_scale=0.3)


def _states(P, seed=0):
    rng = np.random.default_rng(seed)
    return (2.3 + 3.6 * rng.normal(size=(D, P))).astype(np.float32)


@pytest.mark.parametrize("P", [256, 1000])
def test_fused_flow_matches_gemm_path_and_oracle(ctx, torch_gpu, orc, P):
    torch = torch_gpu
    net = capi.MLP(ctx, [41, 256, 256, 256, 40], seed=11)
    norm, F = _norm(), 8.5
    X = _states(P, seed=P)
    Xd = torch.from_numpy(X).cuda()
    out = net.surrogate_flow(norm, F, Xd).cpu().numpy()
    U = np.concatenate([(X.T - np.float32(2.3)) * np.float32(1 / np.float32(3.6)),
                        np.full((P, 1), 0.5, np.float32)], axis=1)
    U = np.ascontiguousarray(U, dtype=np.float32)
    y_gemm = net.forward(torch.from_numpy(U).cuda()).cpu().numpy()
    y_fused = (out - X).T / np.float32(0.3)
    y_orc = orc.mlp_forward(net.dims, net.get_params().astype(np.float64), U.astype(np.float64),
                            bf16=True)
    scale = np.abs(y_orc).max()
    e1 = np.abs(y_fused - y_gemm).max() / scale
    e2 = np.abs(y_fused - y_orc).max() / scale
    print("P", P, "fused vs gemm", e1, "fused vs oracle", e2, flush=True)
    assert e1 < 5e-3 and e2 < 5e-3
    net.close()


def _filter(ctx, P, T, y, mean0, seed=5, ess_rel=0.0):
    m = capi.make_model("l96", d=D, precision=capi.F32, F=8.0, noise_sd=0.1, obs_sd=1.0,
                        init_sd=1.0)
    pf = capi.ParticleFilter(ctx, m, P, T, 0.05, seed, ess_rel=ess_rel)
    pf.set_observations(y)
    pf.init(mean0)
    return pf


def test_filter_step_is_flow_noise_and_density(ctx, torch_gpu, orc):
    torch = torch_gpu
    from libbi_amd import data
    P, T, seed = 1000, 3, 5
    mean0 = data.l96_spinup(ctx, d=D)
    gm = capi.make_model("l96", d=D, precision=capi.F32)
    _, y = data.simulate(ctx, gm, mean0, T, 0.05, seed=9)
    net = capi.MLP(ctx, [41, 256, 256, 256, 40], seed=12)
    norm = _norm()
    pf = _filter(ctx, P, T, y, mean0, seed=seed)
    pf.set_surrogate(net, norm)
    Xd, ld, _ = pf.state()
    x = Xd[:, :P].clone()
    lws_ref = np.zeros(P)
    om = orc.make_model("l96", d=D)
    for k in range(T):
        pf.step(1)
        flow = net.surrogate_flow(norm, 8.0, x.contiguous()).cpu().numpy().astype(np.float64)
        z = np.stack([orc.normals(seed, p, k + 1, orc.TAG_NOISE, D, bits=24) for p in range(P)],
                     axis=1)
        x_ref = flow + 0.1 * z
        Xd, ld, lws = pf.state()
        got = Xd[:, :P].cpu().numpy().astype(np.float64)
        np.testing.assert_allclose(got, x_ref, rtol=0, atol=2e-5)
        lws_ref = orc.obs_logdensity(om, y[k], got, lws_ref)
        np.testing.assert_allclose(lws.cpu().numpy()[:P], lws_ref, rtol=1e-9, atol=1e-9)
        x = Xd[:, :P].clone()
    pf.close()
    net.close()


@pytest.mark.parametrize("other_stream", [False, True])
def test_inference_weights_follow_the_parameters(ctx, torch_gpu, other_stream):
    """New parameters reach the fused kernel at the next call, also from a context on
    another stream than the network's: equal to a network that had them from the start."""
    torch = torch_gpu
    norm = capi.SurrogateNorm(x_shift=2.3, x_scale=3.6, par_shift=8.0, par_scale=1.0,
                              dx_scale=0.3)
    X = torch.randn((40, 1000), device="cuda")
    new = capi.MLP(ctx, surrogate.DIMS, seed=9)
    net = capi.MLP(ctx, surrogate.DIMS, seed=4)
    old = net.surrogate_flow(norm, 8.1, X)
    user = net
    s = torch.cuda.Stream()
    if other_stream:
        torch.cuda.synchronize()  # X was made on torch's stream
        c2 = capi.Context(0, stream=s)
        user = capi.MLP.__new__(capi.MLP)
        user.ctx, user.dims, user.h = c2, net.dims, net.h
    first = user.surrogate_flow(norm, 8.1, X)
    net.set_params(new.get_params())
    second = user.surrogate_flow(norm, 8.1, X)
    torch.cuda.synchronize()
    ref = new.surrogate_flow(norm, 8.1, X)
    torch.cuda.synchronize()
    assert torch.equal(second, ref) and torch.equal(first, old)
    assert not torch.equal(first, ref)
    if other_stream:
        user.h = None
        c2.close()
    net.close()
    new.close()


def test_layout_waits_for_the_reads_of_other_streams(ctx, torch_gpu):
    """Flows of many particles queued on two other streams, then new parameters and a
    flow on the network's own stream at once: the first flows still see the old weights."""
    torch = torch_gpu
    norm = _norm()
    new = capi.MLP(ctx, surrogate.DIMS, seed=9)
    net = capi.MLP(ctx, surrogate.DIMS, seed=4)
    X = torch.randn((40, 1 << 20), device="cuda")
    torch.cuda.synchronize()
    old, ref = net.surrogate_flow(norm, 8.1, X), new.surrogate_flow(norm, 8.1, X)
    p = new.get_params()
    ctx.sync()
    streams = [torch.cuda.Stream() for _ in range(2)]
    users = [capi.Context(0, stream=s) for s in streams]
    outs = [torch.empty_like(X) for _ in range(6)]
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        capi.check(capi.lib().bihip_surrogate_flow(
            users[i % 2].h, net.h, ctypes.byref(norm), 8.1, capi.ptr(X), capi.ptr(out),
            X.shape[1], X.shape[1]))
    net.set_params(p)
    last = net.surrogate_flow(norm, 8.1, X)
    torch.cuda.synchronize()
    assert all(torch.equal(out, old) for out in outs)
    assert torch.equal(last, ref) and not torch.equal(old, ref)
    for c in users:
        c.close()
    net.close()
    new.close()


def test_filter_keeps_the_network_it_was_given(ctx, torch_gpu):
    """The network is read when it is attached: new parameters reach neither the weights
    nor the biases of a filter that already has it."""
    m = capi.make_model("l96", d=40, precision=capi.F32, init_sd=0.3)
    y = np.random.default_rng(2).normal(2.3, 3.6, (4, 20))
    got = []
    for change in (False, True):
        net = capi.MLP(ctx, surrogate.DIMS, seed=4)
        pf = capi.ParticleFilter(ctx, m, 3000, 4, 0.05, 7)
        pf.set_observations(y)
        pf.set_surrogate(net, _norm())
        pf.init(np.full(40, 2.0))
        pf.step(1)
        if change:
            net.set_params(0.5 * net.get_params())
        pf.step(3)
        got.append((pf.outputs()["logIncrements"], pf.state()[0][:, :3000].cpu().numpy()))
        pf.close()
        net.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


def test_layout_refuses_a_captured_stream(ctx, torch_gpu):
    """A replay would not lay out the weights that the network has by then."""
    torch = torch_gpu
    s = torch.cuda.Stream()
    c2 = capi.Context(0, stream=s)
    net = capi.MLP(c2, surrogate.DIMS, seed=4)
    X = torch.randn((40, 64), device="cuda")
    out = torch.empty_like(X)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        graph.capture_begin()
        rc = capi.lib().bihip_surrogate_flow(c2.h, net.h, ctypes.byref(_norm()), 8.1,
                                             capi.ptr(X), capi.ptr(out), 64, 64)
        out.add_(1.0)  # a graph of something
        graph.capture_end()
    assert rc != capi.OK
    torch.cuda.synchronize()
    a = net.surrogate_flow(_norm(), 8.1, X)  # the network is as before
    c2.sync()
    ref = capi.MLP(ctx, surrogate.DIMS, seed=4)
    b = ref.surrogate_flow(_norm(), 8.1, X)
    ctx.sync()
    assert torch.equal(a, b)
    ref.close()
    net.close()
    c2.close()


@pytest.mark.parametrize("P", [1, 31, 33, 256, 257, 600])
def test_fused_networks_at_ragged_particle_counts(ctx, torch_gpu, P):
    """Particles around a wave's 32 and a workgroup's 256: the same bits as in a larger
    batch, the columns past the last particle untouched."""
    torch = torch_gpu
    big, ld = 700, 700
    norm = _norm()
    net = capi.MLP(ctx, surrogate.DIMS, seed=4)
    X = torch.from_numpy(_states(big, seed=3)).cuda()
    ref = net.surrogate_flow(norm, 8.1, X)
    out = torch.full_like(X, 7.0)
    capi.check(capi.lib().bihip_surrogate_flow(ctx.h, net.h, ctypes.byref(norm), 8.1, capi.ptr(X),
                                               capi.ptr(out), ld, P))
    assert torch.equal(out[:, :P], ref[:, :P]) and bool((out[:, P:] == 7.0).all())
    net.close()

    gnorm = capi.GuidedNorm(x_shift=2.3, x_scale=3.6, innov_scale=1.0, par_shift=8.0,
                            par_scale=1.0)
    gnet = capi.MLP(ctx, guided.DIMS, seed=5)
    Phi = 2.3 + 3.6 * torch.randn((200, big), device="cuda")
    y = torch.randn(100, dtype=torch.float64, device="cuda")
    got = []
    for n in (big, P):
        Z, inc = Phi.clone(), torch.full((big,), 7.0, dtype=torch.float64, device="cuda")
        capi.check(capi.lib().bihip_guided_propose(
            ctx.h, gnet.h, ctypes.byref(gnorm), 8.2, capi.ptr(Z), ld, n, capi.ptr(y), 5, 2, 3,
            0.1, 1.0, capi.ptr(inc)))
        got.append((Z, inc))
    (Za, ia), (Zb, ib) = got
    assert torch.equal(Zb[:, :P], Za[:, :P]) and torch.equal(Zb[:, P:], Phi[:, P:])
    assert torch.equal(ib[:P], ia[:P]) and bool((ib[P:] == 7.0).all())
    gnet.close()
