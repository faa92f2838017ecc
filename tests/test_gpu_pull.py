"""Networks stepped over the whole chip, whose neurons count their own events
(brian2_amd/chip.py), against the staged launches (tile given), bit for bit."""
import numpy as np
import pytest

from test_gpu_resident import _const_spec

pytestmark = pytest.mark.gpu

E = ("ge", "+=", 1.62e-3)
I = ("gi", "+=", -9e-3)
CASES = {
    "one neuron": (1, "double", [((0, 1), (0, 1)) + E + (1.0,)], "start"),
    "a word": (64, "double", [((0, 64), (0, 64)) + E + (0.5,), ((0, 64), (0, 64)) + I + (0.2,)], None),
    "a word and one": (65, "float", [((3, 65), (0, 65)) + E + (0.5,), ((0, 7), (1, 60)) + I + (1.0,)], "end"),
    "a chunk of words": (4096, "double", [((0, 3000), (0, 4096)) + E + (0.01,), ((3000, 4096), (0, 4096)) + I + (0.01,)],
                         "start"),
    "a chunk and one": (4097, "float", [((0, 4097), (7, 4090)) + E + (0.01,)], None),
    "the largest": (16384, "double", [((0, 13000), (0, 16384)) + E + (0.004,), ((13000, 16384), (0, 16384)) + I + (0.004,)],
                    "end"),
    "one variable, a pathway without synapses": (700, "double", [
        ((0, 700), (0, 700), "ge", "+=", 1.1e-3, 0.03), ((0, 300), (0, 700), "ge", "*=", 0.9, 0.02),
        ((0, 700), (0, 700)) + I + (0.0,), ((200, 700), (0, 400), "ge", "-=", 1e-4, 0.03)], None),
}


def _run(n, float_t, paths, state, model="cuba", twice=False, **options):
    from brian2_amd import (Model, Network, NeuronGroup, PopulationRateMonitor, SpikeMonitor, StateMonitor, Synapses)

    rng = np.random.default_rng(5)
    G = NeuronGroup(n, Model.load(model), float_t=float_t, name="g")
    G.v = -0.06 + 0.02 * rng.random(n) if model == "cuba" else -0.06 + 0.05 * rng.random(n)
    G.lastspike = np.where(rng.random(n) < 0.3, -3.3e-3 * rng.random(n), -1e4)
    syn = []
    for k, (src, tgt, var, op, value, p) in enumerate(paths):
        a, b = G[src[0]:src[1]], G[tgt[0]:tgt[1]]
        S = Synapses(a, b, _const_spec(var, op, value), name=f"s{k}")
        i, j = np.nonzero(rng.random((a.N, b.N)) < p)
        S.connect(np.append(i, i[:1]), np.append(j, j[:1])) if twice else S.connect(i, j)
        syn.append(S)
    spikes, rate = SpikeMonitor(G[n // 3:]), PopulationRateMonitor(G[:max(1, n // 2)])
    mons = [StateMonitor(G, ["v", "ge"], record=sorted({0, n // 2, n - 1}), when=state)] if state else []
    net = Network(G, *syn, spikes, rate, *mons, dt=1e-4, **options)
    for k in (1, 40, 19):
        net.run(k)
    net.store()
    net.run(30)
    net.restore()
    net.run(20)
    net.run(10, dt=5e-5)
    out = [G.get(v) for v in G.vars] + [np.array([s.n_events for s in syn])]
    return G, out + [spikes.i, spikes.step, spikes.count, rate.count] + [m.values() for m in mons]


@pytest.mark.parametrize("name", sorted(CASES))
def test_pulled_events_equal_the_staged_launches(name, monkeypatch):
    from brian2_amd import resident

    monkeypatch.setattr(resident.GroupStep, "takes", classmethod(lambda *a: False))
    G, got = _run(*CASES[name])
    H, want = _run(*CASES[name], tile=256)
    assert G.pull is not None and H.pull is None
    assert CASES[name][0] == 1 or want[0].std() > 0
    for x, y in zip(got, want):
        assert np.array_equal(x, y)


def test_cobahh_pulls_and_what_is_not_taken():
    """The example with exponentials by default; pairs with two synapses and launch shapes stay."""
    paths = [((0, 900), (0, 1100), "ge", "+=", 6e-9, 0.02), ((900, 1100), (0, 1100), "gi", "+=", 6.7e-8, 0.02)]
    G, got = _run(1100, "double", paths, "start", model="cobahh")
    H, want = _run(1100, "double", paths, "start", model="cobahh", tile=128)
    assert G.pull is not None and H.pull is None
    assert len(want[-4]) > 0
    for x, y in zip(got, want):
        assert np.array_equal(x, y)
    assert _run(1100, "double", paths, None, model="cobahh", twice=True)[0].pull is None


def test_parts_of_an_update():
    """The parts that waves may take read nothing that the update has written before, and
    temporaries that read each other stay together."""
    from brian2_amd.kernels import CodeSpec, split_update

    def st(var, op, expr):
        return dict(var=var, op=op, expr=expr, dtype="float64")

    code = [st("a", ":=", "exp(x)"), st("b", ":=", "exp(a) + x"), st("c", ":=", "y ** 3"), st("x", "=", "b"),
            st("d", ":=", "exp(x)"), st("e", ":=", "c + exp(z)"), st("f", ":=", "z + y"), st("y", "=", "d + e + f")]
    spec = CodeSpec({"name": "u", "template": "stateupdate", "owner": "g", "variables": {}, "indices": {},
                     "blocks": {"None": {"scalar": [], "vector": code, "conditional_write": {}}}})
    assert split_update(spec, 4) == [[0, 1], [2, 5]]
    assert split_update(spec, 1) == [[0, 1, 2, 5]]


@pytest.mark.parametrize("n, delay, options, form", [(300, 0.0, {}, "chip"), (300, 0.0, {"tile": 256}, "staged"),
                                                     (300, 0.0, {"tile": 64, "npt": 2}, "staged"),
                                                     (6000, 3e-4, {}, "fused")])
def test_a_reset_that_follows_the_events_has_its_steps_time(n, delay, options, form):
    """A reset that writes a variable of the pathways runs behind them; the time that it reads
    is that of the spike, in the steps of a run and at its end."""
    from brian2_amd import Model, Network, NeuronGroup, SpikeMonitor, Synapses

    rng = np.random.default_rng(4)
    m = Model.load("cuba")
    rs = m.group["reset"]
    rs.vector = rs.vector + [dict(var="ge", op="=", expr="0.0", dtype="float64"),
                             dict(var="tlast", op="=", expr="t", dtype="float64")]
    rs.variables = dict(rs.variables, t=m.group["stateupdate"].variables["t"])
    G = NeuronGroup(n, m, name="g", variables={"tlast": "float64"})
    G.v = -0.06 + 0.02 * rng.random(n)
    G.tlast = -1.0
    S = Synapses(G, G, _const_spec(*E))
    S.connect(*np.nonzero(rng.random((n, n)) < 30.0 / n))
    S.set_delay(delay)
    mon = SpikeMonitor(G)
    net = Network(G, S, mon, dt=1e-4, **options)
    want = np.full(n, -1.0)
    for k in (1, 60, 139):
        net.run(k)
        want[mon.i] = mon.step * 1e-4
        assert (G.pull is not None) == (form == "chip") and (getattr(G, "fused", None) is not None) == (form == "fused")
        assert np.array_equal(G.get("tlast"), want)
        assert np.array_equal(G.get("lastspike")[want >= 0], want[want >= 0])
    assert (want >= 0).sum() > n // 4 and (want == 199 * 1e-4).any() == (199 in mon.step)


def _waiting_network(form, **options):
    from brian2_amd import Model, Network, NeuronGroup, PopulationRateMonitor, SpikeMonitor, StateMonitor, Synapses, synth

    if form == "chip":
        c = synth.cobahh_network(N=1000, record=[3, 70], network_options=options)
        return c["net"], c["G"], c["mon"], c["state"]
    rng = np.random.default_rng(2)
    m = Model.load("gap")
    G = NeuronGroup(100, m)
    G.v = 1.3 * rng.random(100)
    S = Synapses(G, G, summed={"Igap": m.summed["Igap"]})
    S.connect(np.repeat(np.arange(100), 100), np.tile(np.arange(100), 100))
    S.set("w", 0.06 * rng.random(10000))
    mon, state = SpikeMonitor(G), StateMonitor(G, ["v"], record=[3, 70])
    return Network(G, S, mon, state, PopulationRateMonitor(G), dt=1e-4, **options), G, mon, state


@pytest.mark.parametrize("form", ["chip", "sums"])
def test_a_launch_whose_workgroups_do_not_all_run_changes_nothing(form, monkeypatch):
    """A launch that misses a workgroup (one more is expected than there are, few polls) ends
    without a step and is made again; after too many of them a run fails, and the next goes on."""
    import torch

    from brian2_amd import chip, runtime
    from brian2_amd._lib import HipBrianError

    def results(x):
        net, G, mon, state = x
        return [G.get(v) for v in G.vars] + [mon.i, mon.step, mon.count, state.values(), state.t_]

    a, b = _waiting_network(form), _waiting_network(form)
    for x in (a, b):
        x[0].run(60)
    launches, zero = [], torch.Tensor.zero_

    def run(x):
        if x is b[0].in_launch.xch:
            launches.append(1)
            zero(x)
            if len(launches) in missing:
                x[-2], x[-1] = 1, chip.SPINS - 3
            return x
        return zero(x)

    a[0].run(50)
    a[0].run(70)
    monkeypatch.setattr(torch.Tensor, "zero_", run)
    missing = {1, 2, 4}
    b[0].run(50)
    b[0].run(70)
    assert len(launches) == 5
    assert all(np.array_equal(x, y) for x, y in zip(results(a), results(b)))
    monkeypatch.setattr(runtime, "TRIES", 2)
    before = [b[1].get(v) for v in b[1].vars] + [b[2].i, b[0].t_step]
    missing = set(range(100))
    with pytest.raises(HipBrianError, match="did not come to run"):
        b[0].run(40)
    assert all(np.array_equal(x, y) for x, y in zip(before, [b[1].get(v) for v in b[1].vars] + [b[2].i, b[0].t_step]))
    missing = set()
    a[0].run(40)
    b[0].run(40)
    assert all(np.array_equal(x, y) for x, y in zip(results(a), results(b)))


@pytest.mark.parametrize("form", ["chip", "sums"])
def test_networks_whose_workgroups_do_not_fit_at_once(form, monkeypatch):
    """As many workgroups as the device says it runs at once, and no more."""
    from brian2_amd import runtime

    x, y = _waiting_network(form), _waiting_network(form)
    x[0].run(120)
    assert x[0].in_launch is not None
    assert x[0].device.together(x[0].in_launch.fn, x[0].in_launch.threads) % x[0].device.n_cu == 0
    monkeypatch.setattr(runtime.Device, "together", lambda self, fn, threads: x[0].in_launch.grid - 1)
    y[0].run(120)
    assert y[0].in_launch is None or y[0].resident is not None
    assert len(x[2].i) > 0 and np.array_equal(x[2].i, y[2].i) and np.array_equal(x[2].step, y[2].step)
    assert all(np.array_equal(x[1].get(v), y[1].get(v)) for v in x[1].vars)
