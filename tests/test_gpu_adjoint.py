"""The differentiable LIF network on the device: forward parity with Brian, the
adjoint against autograd of the unrolled tensor reference, and against fp64
central finite differences at perturbations that create or delete no spike."""
import numpy as np
import pytest

import oracle_py as O

pytestmark = pytest.mark.gpu


def _net(trials=2, wt="float"):
    from brian2_amd.adjoint import LIFNetwork

    return LIFNetwork(trials=trials, weight_dtype=wt)


def test_forward_bitexact_vs_brian():
    z, meta = O.load_golden("lif")
    net = _net(meta["trials"])
    loss, saved = net.forward(net.w_in0, net.w_rec0, net.c["tau_m"], net.c["tau_s"], record_spikes=True)
    for b in range(meta["trials"]):
        i, s = saved["spikes"][b]
        sel = z["trial"] == b
        assert len(i) == sel.sum()
        assert np.array_equal(i, z["i"][sel]) and np.array_equal(s, z["step"][sel])
        assert np.array_equal(saved["v"][b].cpu().numpy(), z["final"][b][0])
        assert np.array_equal(saved["I"][b].cpu().numpy(), z["final"][b][1])
    assert np.isfinite(loss)


def _reference(net, trials):
    import torch

    from lif_reference import reference_loss

    inp = O.lif_inputs(trials)
    sc, _ = net._scalars(net.c["tau_m"], net.c["tau_s"])
    lio = tuple(sc[f"_lio_{k}"] for k in (1, 2, 3, 4))
    w_in = torch.tensor(net.w_in0.cpu().numpy().astype(np.float64), requires_grad=True)
    w_rec = torch.tensor(net.w_rec0.cpu().numpy().astype(np.float64), requires_grad=True)
    tm = torch.tensor(net.c["tau_m"], dtype=torch.float64, requires_grad=True)
    ts = torch.tensor(net.c["tau_s"], dtype=torch.float64, requires_grad=True)
    loss, fs, raster = reference_loss(inp, inp["trains"], inp["v0"], w_in, w_rec, tm, ts, net.c, lio_values=lio)
    loss.backward()
    return float(loss), w_in.grad.numpy(), w_rec.grad.numpy(), float(tm.grad), float(ts.grad), raster


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def test_adjoint_equals_autograd_of_the_tensor_reference():
    import torch

    from brian2_amd.adjoint import lif_loss

    net = _net(2, "double")
    w_in = net.w_in0.clone().requires_grad_(True)
    w_rec = net.w_rec0.clone().requires_grad_(True)
    tm = torch.tensor(net.c["tau_m"], dtype=torch.float64, requires_grad=True)
    ts = torch.tensor(net.c["tau_s"], dtype=torch.float64, requires_grad=True)
    loss = lif_loss(net, w_in, w_rec, tm, ts)
    loss.backward()
    ref_loss, g_in, g_rec, g_m, g_s, _ = _reference(net, 2)
    print(f"loss {float(loss)!r} reference {ref_loss!r}; dL/dtau_m {float(tm.grad)!r} vs {g_m!r}; "
          f"dL/dtau_s {float(ts.grad)!r} vs {g_s!r}", flush=True)
    assert abs(float(loss) - ref_loss) <= 1e-11 * abs(ref_loss)
    assert _rel(w_in.grad.cpu().numpy(), g_in) < 1e-9
    assert _rel(w_rec.grad.cpu().numpy(), g_rec) < 1e-9
    assert abs(float(tm.grad) - g_m) <= 1e-9 * abs(g_m)
    assert abs(float(ts.grad) - g_s) <= 1e-9 * abs(g_s)


def test_adjoint_equals_central_finite_differences():
    """fp64 central differences at perturbations that leave every spike in place:
    for each parameter the largest step of a short list (relative 1e-5 .. 1e-7 for
    the time constants, 1e-2 .. 1e-4 sigma for weights) whose +h and -h runs
    reproduce the unperturbed spike raster exactly."""
    net = _net(2, "double")
    w_in, w_rec = net.w_in0.clone(), net.w_rec0.clone()
    tm, ts = net.c["tau_m"], net.c["tau_s"]
    loss0, saved = net.forward(w_in, w_rec, tm, ts, record_spikes=True)
    g_in, g_rec, g_m, g_s = net.backward(saved)
    g_in, g_rec = g_in.cpu().numpy(), g_rec.cpu().numpy()
    ref = saved["spikes"]

    def L(wi, wr, m, s):
        loss, sv = net.forward(wi, wr, m, s, record_spikes=True)
        same = all(np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) for a, b in zip(sv["spikes"], ref))
        return loss, same

    def fd(make, steps):
        for h in steps:
            (lp, sp), (lm, sm) = L(*make(h)), L(*make(-h))
            if sp and sm:
                return (lp - lm) / (2 * h), h
        return None, None

    checks = []
    checks.append(("tau_m",) + fd(lambda h: (w_in, w_rec, tm + h, ts), [r * tm for r in (1e-5, 1e-6, 1e-7)]) + (g_m,))
    checks.append(("tau_s",) + fd(lambda h: (w_in, w_rec, tm, ts + h), [r * ts for r in (1e-5, 1e-6, 1e-7)]) + (g_s,))
    sig = net.inp["sigma"]
    for name, g, which in (("w_in", g_in, 0), ("w_rec", g_rec, 1)):
        for e in np.argsort(-np.abs(g))[:3]:
            def make(h, e=int(e), which=which):
                w = [w_in.clone(), w_rec.clone()]
                w[which][e] += h
                return w[0], w[1], tm, ts
            checks.append((f"{name}[{e}]",) + fd(make, [r * sig for r in (1e-2, 1e-3, 1e-4)]) + (float(g[e]),))
    for name, d, h, adj in checks:
        print(f"{name}: finite difference {d!r} (step {h!r}), adjoint {adj!r}", flush=True)
        assert d is not None, f"{name}: every step changed a spike"
        assert abs(d - adj) <= 1e-6 * abs(adj), name


def test_full_configuration_is_deterministic():
    """256 trials, fp32 weights: forward + backward twice give identical results."""
    import torch

    net = _net(256, "float")
    outs = []
    for _ in range(2):
        loss, saved = net.forward(net.w_in0, net.w_rec0, net.c["tau_m"], net.c["tau_s"])
        g = net.backward(saved)
        outs.append((loss, g[0].cpu().numpy(), g[1].cpu().numpy(), g[2], g[3]))
        torch.cuda.synchronize()
    a, b = outs
    assert np.isfinite(a[0]) and a[0] == b[0]
    assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2]) and a[3] == b[3] and a[4] == b[4]
    assert np.isfinite(a[1]).all() and np.abs(a[2]).max() > 0


@pytest.mark.parametrize("n, n_in, p, rate, steps, every, wt", [
    (64, 1, 0.1, 500.0, 60, 20, "double"),      # one wave, one input, blocks of 8 and a rest of 4
    (65, 64, 1e-9, 500.0, 50, 50, "float"),     # a second word of one neuron; no synapses
    (300, 65, 1.0, 300.0, 70, 7, "double"),    # rows longer than their pieces, an interval within a block
    (513, 200, 0.1, 1500.0, 60, 30, "float"),  # many events: several per word, row and block
    (1024, 1024, 0.05, 100.0, 40, 1, "float"),  # the largest
])
def test_shapes_at_the_edges_of_words_blocks_and_batches(n, n_in, p, rate, steps, every, wt):
    """Loss and gradients against autograd of the tensor reference (both double beyond the
    weights' rounding; sums of at most 1e5 terms, so 1e-9)."""
    import torch

    from brian2_amd.adjoint import LIF, LIFNetwork
    from lif_reference import reference_loss

    c = dict(LIF, N=n, NE=n * 4 // 5, n_in=n_in, p=p, rate_lo=rate / 2, rate_hi=rate, n_steps=steps, tau_m=0.004, bias=0.012)
    net = LIFNetwork(trials=3, config=c, weight_dtype=wt, ckpt_every=every)
    loss, saved = net.forward(net.w_in0, net.w_rec0, c["tau_m"], c["tau_s"])
    g_in, g_rec, g_m, g_s = net.backward(saved)
    sc, _ = net._scalars(c["tau_m"], c["tau_s"])
    leaf = lambda x: torch.tensor(x, dtype=torch.float64, requires_grad=True)  # noqa: E731
    w_in, w_rec = leaf(net.w_in0.cpu().numpy().astype(np.float64)), leaf(net.w_rec0.cpu().numpy().astype(np.float64))
    tm, ts = leaf(c["tau_m"]), leaf(c["tau_s"])
    ref, _, raster = reference_loss(net.inp, O.lif_inputs(3, c=c)["trains"], net.inp["v0"], w_in, w_rec, tm, ts, c,
                                    lio_values=tuple(sc[f"_lio_{k}"] for k in (1, 2, 3, 4)))
    ref.backward()
    assert raster.sum() > 3 * n // 10
    assert abs(loss - float(ref)) <= 1e-11 * abs(float(ref))
    for got, want in ((g_in, w_in), (g_rec, w_rec)):
        got = got.cpu().numpy()
        assert got.shape == tuple(want.shape)
        if len(got) and want.grad is not None and float(want.grad.abs().max()) > 0:
            assert _rel(got, want.grad.numpy()) < 1e-9
    assert abs(g_m - float(tm.grad)) <= 1e-9 * abs(float(tm.grad))
    assert abs(g_s - float(ts.grad)) <= 1e-9 * abs(float(ts.grad))


@pytest.mark.parametrize("n, every, wt", [(65, 7, "float"), (513, 25, "double"), (1000, 100, "float")])
def test_kept_and_recomputed_states_give_the_same_gradients(n, every, wt, monkeypatch):
    """The states at the blocks' starts from the forward pass, and recomputed from the
    intervals' checkpoints (as for runs whose states would be too large to keep)."""
    from brian2_amd import adjoint

    c = dict(adjoint.LIF, N=n, NE=n * 4 // 5, n_steps=every * 4, tau_m=0.004, bias=0.012, rate_hi=400.0)
    out = []
    for keep in (True, False):
        if not keep:
            monkeypatch.setattr(adjoint, "KEEP_BYTES", 0)
        net = adjoint.LIFNetwork(trials=2, config=c, weight_dtype=wt, ckpt_every=every)
        assert net.keep == keep
        loss, saved = net.forward(net.w_in0, net.w_rec0, c["tau_m"], c["tau_s"])
        g = net.backward(saved)
        out.append([np.float64(loss), g[0].cpu().numpy(), g[1].cpu().numpy(), g[2], g[3]])
    assert np.abs(out[0][2]).max() > 0
    assert all(np.array_equal(a, b) for a, b in zip(*out))


def _leaves(net):
    import torch

    w = [x.clone().requires_grad_(True) for x in (net.w_in0, net.w_rec0)]
    return w + [torch.tensor(net.c[k], dtype=torch.float64, requires_grad=True) for k in ("tau_m", "tau_s")]


def test_losses_alive_together_hold_bounded_memory():
    """Losses that are summed before their backward pass: what they hold beside their weights stays
    within 4 GiB; a loss without a backward pass holds nothing and keeps no states on the way."""
    import torch

    from brian2_amd import adjoint

    net = adjoint.LIFNetwork(trials=64)
    states = 16 * 64 * 1000 * 2000 // 8  # of the blocks of the backward pass
    leaves = _leaves(net)
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    with torch.no_grad():
        a = adjoint.lif_loss(net, *leaves)
    b = adjoint.lif_loss(net, *(x.detach() for x in leaves))
    assert torch.cuda.max_memory_allocated() - before < states // 4
    assert torch.cuda.memory_allocated() - before < 1 << 20
    losses = [adjoint.lif_loss(net, *leaves) for _ in range(24)]
    assert float(a) == float(b) == float(losses[0]) == float(losses[-1])
    assert torch.cuda.memory_allocated() - before < (4 << 30) + len(losses) * (8 << 20)
    first, last = (torch.autograd.grad(x, leaves) for x in (losses[0], losses[-1]))
    assert all(torch.equal(x, y) for x, y in zip(first, last)) and float(last[1].abs().max()) > 0
    torch.autograd.backward([sum(losses)])
    assert all(torch.allclose(x.grad.double(), len(losses) * y.double(), rtol=1e-5, atol=0.0)
               for x, y in zip(leaves, first))
    del losses
    assert torch.cuda.memory_allocated() - before < 32 << 20


@pytest.mark.parametrize("n, steps, every, wt", [(65, 56, 7, "float"), (300, 96, 8, "float"), (513, 100, 25, "double")])
def test_every_form_of_what_is_held_gives_the_same_gradients(n, steps, every, wt):
    """The blocks' states, the intervals' states and a second simulation; the room that a loss
    took is there again when it is gone."""
    import torch

    from brian2_amd import adjoint

    c = dict(adjoint.LIF, N=n, NE=n * 4 // 5, n_steps=steps, tau_m=0.004, bias=0.012, rate_hi=400.0)
    net = adjoint.LIFNetwork(trials=3, config=c, weight_dtype=wt, ckpt_every=every)
    net.keep_bytes = net._bytes(net.sub) + net._bytes(net.C)
    leaves = _leaves(net)
    with torch.no_grad():
        values = [float(adjoint.lif_loss(net, *leaves))]
    for _ in range(2):
        losses = [adjoint.lif_loss(net, *leaves) for _ in range(4)]
        held = [x.grad_fn.saved["every"] for x in losses]
        # (an interval of one block has the same states in both forms)
        assert held == [net.sub, net.sub if net.sub >= every else every, 0, 0]
        values += [float(x) for x in losses]
        with torch.no_grad():
            for x in leaves[:2]:  # as an optimizer's step between the passes
                x.mul_(2.0)
        grads = [torch.autograd.grad(x, leaves) for x in reversed(losses)]
        with torch.no_grad():
            for x in leaves[:2]:
                x.mul_(0.5)
        for g in grads[1:]:
            assert all(torch.equal(x, y) for x, y in zip(g, grads[0]))
        assert float(grads[0][1].abs().max()) > 0
        del losses
    assert len(set(values)) == 1


@pytest.mark.parametrize("rates, same_as", [((-50.0, -1.0), (0.0, 0.0)), ((float("nan"), 1.0), (0.0, 0.0)),
                                            ((1.5e4, 3e7), (1e4, 1e4))])
def test_rates_outside_of_a_probabilitys_range(rates, same_as):
    """A draw is compared with rate dt: a rate below 0 or NaN never spikes, one of 1 / dt and more
    always."""
    from brian2_amd import adjoint

    out = []
    for lo, hi in (rates, same_as):
        c = dict(adjoint.LIF, N=100, NE=80, n_steps=200, rate_lo=lo, rate_hi=hi, tau_m=0.004, bias=0.012)
        net = adjoint.LIFNetwork(trials=2, config=c)
        loss, saved = net.forward(net.w_in0, net.w_rec0, c["tau_m"], c["tau_s"], record_spikes=True)
        out.append([np.float64(loss)] + [x for pair in saved["spikes"] for x in pair])
    assert len(out[0][1]) > 0 and all(np.array_equal(x, y) for x, y in zip(*out))
