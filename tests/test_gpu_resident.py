"""Small networks without delays, stepped by one workgroup (brian2_amd/resident.py),
against the staged launches of the same networks (tile given), bit for bit."""
import numpy as np
import pytest

from test_gpu_kats import onpre_spec

pytestmark = pytest.mark.gpu

STATE = ("v", "ge", "gi", "lastspike", "not_refractory")


def _const_spec(var, op, value):
    """on_pre='<var> <op> <value>' as Brian's statements."""
    s = onpre_spec(repr(value))
    s.vector = [dict(s.vector[0], var=var, op=op)]
    s.variables[var] = dict(s.variables["v"])
    s.indices[var] = "_postsynaptic_idx"
    return s


def _network(n, float_t, paths, monitors, seed=3, **options):
    """CUBA neurons, about half of them above threshold in the first step."""
    from brian2_amd import (Model, Network, NeuronGroup, PopulationRateMonitor, SpikeMonitor, StateMonitor, Synapses)

    rng = np.random.default_rng(seed)
    G = NeuronGroup(n, Model.load("cuba"), float_t=float_t, name="g")
    G.v = -0.06 + 0.02 * rng.random(n)
    G.lastspike = np.where(rng.random(n) < 0.3, -3.3e-3 * rng.random(n), -1e4)
    syn = []
    for k, (src, tgt, var, op, value, p) in enumerate(paths):
        a, b = G[src[0]:src[1]], G[tgt[0]:tgt[1]]
        S = Synapses(a, b, _const_spec(var, op, value), name=f"s{k}")
        i, j = np.nonzero(rng.random((a.N, b.N)) < p)
        twice = rng.random(len(i)) < 0.1  # some pairs with two synapses
        S.connect(np.concatenate([i, i[twice]]), np.concatenate([j, j[twice]]))
        syn.append(S)
    mons = {}
    if "spikes" in monitors:
        mons["spikes"] = SpikeMonitor(G)
    if "some" in monitors:
        mons["spikes"] = SpikeMonitor(G[n // 3:n - n // 4])
    if "rate" in monitors:
        mons["rate"] = PopulationRateMonitor(G[:max(1, n // 2)])
    if "state" in monitors:
        mons["state"] = StateMonitor(G, ["v", "ge"], record=sorted({0, n // 2, n - 1}))
    if "lastspike" in monitors:
        mons["state"] = StateMonitor(G, ["lastspike", "gi"], record=[0, n - 1])
    net = Network(G, *syn, *mons.values(), dt=1e-4, **options)
    return net, G, syn, mons


def _results(built, pieces):
    net, G, syn, mons = built
    for k in pieces:
        net.run(k)
    out = [G.get(v) for v in STATE] + [np.array([s.n_events for s in syn])]
    if "spikes" in mons:
        out += [mons["spikes"].i, mons["spikes"].step, mons["spikes"].count]
    if "rate" in mons:
        out.append(mons["rate"].count)
    if "state" in mons:
        out.append(mons["state"].values())
    return out


E = ("ge", "+=", 1.62e-3)
I = ("gi", "+=", -9e-3)
CASES = {
    "one neuron": (1, "double", lambda n: [((0, 1), (0, 1)) + E + (1.0,)], ("spikes",)),
    "a wave": (64, "double", lambda n: [((0, n), (0, n)) + E + (0.5,)], ("spikes", "rate", "state")),
    "a wave and one": (65, "float", lambda n: [((0, n), (0, n)) + E + (0.5,), ((0, n), (0, n)) + I + (0.2,)],
                       ("some", "rate")),
    "a workgroup": (1024, "double", lambda n: [((0, 800), (0, n)) + E + (0.05,), ((800, n), (0, n)) + I + (0.05,)],
                    ("spikes", "lastspike")),
    "two per thread": (1025, "float", lambda n: [((0, n), (5, n - 7)) + E + (0.03,)], ("spikes", "state")),
    "ragged": (2999, "double", lambda n: [((0, 2000), (0, n)) + E + (0.02,), ((2000, n), (100, n)) + I + (0.02,)],
               ("some", "rate", "state")),
    "eight per thread": (8192, "double", lambda n: [((0, 6000), (0, n)) + E + (0.004,),
                                                    ((6000, n), (0, n)) + I + (0.004,)], ("spikes",)),
    "one variable, four pathways": (700, "double", lambda n: [
        ((0, n), (0, n), "ge", "+=", 1.1e-3, 0.03), ((0, 300), (0, n), "ge", "*=", 0.9, 0.02),
        ((200, n), (0, 400), "ge", "-=", 1e-4, 0.03), ((0, n), (0, n)) + I + (0.01,)], ("spikes",)),
    "a pathway without synapses": (300, "double", lambda n: [((0, n), (0, n)) + E + (0.0,),
                                                             ((0, n), (0, n)) + I + (0.1,)], ()),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_resident_equals_the_staged_launches(name):
    n, float_t, paths, monitors = CASES[name]
    a = _network(n, float_t, paths(n), monitors)
    b = _network(n, float_t, paths(n), monitors, tile=256)
    got, want = _results(a, (1, 130, 69)), _results(b, (200,))
    assert a[0].resident is not None and b[0].resident is None
    assert n == 1 or want[0].std() > 0
    for x, y in zip(got, want):
        assert np.array_equal(x, y)


def test_resident_store_restore_dt_and_profile():
    """store and restore, a change of dt between runs, profile(): as the staged launches."""
    n, float_t, paths, monitors = CASES["ragged"]
    out = []
    for options in ({}, {"tile": 256}):
        built = _network(n, float_t, paths(n), ("spikes",), **options)
        net, G, syn, mons = built
        net.run(50)
        net.store()
        first = _results(built, (60,))
        net.restore()
        net.profile(60)
        net.run(0)
        assert all(np.array_equal(x, y) for x, y in zip(_results(built, ()), first))
        net.run(40, dt=5e-5)
        net.run(40, dt=1e-4)
        out.append(_results(built, ()) + [mons["spikes"].t_])
    for x, y in zip(*out):
        assert np.array_equal(x, y)


def test_networks_that_are_not_taken():
    """Delays, variables of the synapses, launch shapes and heavy updates keep the staged launches."""
    from brian2_amd import synth

    for c in (synth.cuba_synw_network(N=600, K=20), synth.cuba_network(N=600, network_options={"gather_pairs": 16}),
              synth.cobahh_network(N=1000), synth.cuba_network(N=9000)):
        c["net"].run(2)
        assert c["net"].resident is None


@pytest.mark.parametrize("steps", [2**30 - 1, 2**30, 2**31 - 2, 2**31, 3 * 10**9])
def test_refractory_periods_beyond_32_bits(steps):
    """Neurons that fire once: a period whose steps, or whose release step counted from a
    launch's beginning, take more than 32 bits."""
    from brian2_amd import Model, Network, NeuronGroup, SpikeMonitor, Synapses

    out = []
    for options in ({}, {"tile": 256}):
        m = Model.load("cuba")
        m.group["stateupdate"].scalar[0]["expr"] = f"timestep({steps!r} * dt, dt)"
        G = NeuronGroup(200, m, name="g")
        G.v = np.linspace(-0.06, -0.04, 200)
        G.lastspike = -1e7
        S = Synapses(G, G, _const_spec("ge", "+=", 1.62e-3))
        S.connect(*np.nonzero(np.random.default_rng(1).random((200, 200)) < 0.2))
        mon = SpikeMonitor(G)
        net = Network(G, S, mon, dt=1e-4, **options)
        for k in (100, 1, 99):
            net.run(k)
        assert (net.resident is not None) == (not options)
        out.append([mon.i, mon.step] + [G.get(v) for v in STATE])
    assert len(out[1][0]) > 100 and np.bincount(out[1][0]).max() == 1
    for x, y in zip(*out):
        assert np.array_equal(x, y)
