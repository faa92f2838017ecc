"""Models whose variables have the names that generated code might use itself: the same
results as under their own names, in every form of the steps that holds the state in registers."""
import json
import os
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(name, names):
    """The model with its variables renamed (the generator's names kept apart)."""
    from brian2_amd import Model, runtime

    with open(os.path.join(runtime.SPEC_DIR, f"{name}.json")) as f:
        text = f.read()
    for old, new in names.items():
        text = re.sub(rf"(?<![\w.])(_?){old}((?:_pre|_post)?)(?!\w)", rf"\1{new}\2", text)
    return Model(json.loads(text))


def _group(n, name, names, when, **options):
    from brian2_amd import Network, NeuronGroup, SpikeMonitor, StateMonitor, Synapses, synth

    rng = np.random.default_rng(n)
    m = _model(name, names)
    G = NeuronGroup(n, m, name="g")
    v = names.get("v", "v")
    mons = [SpikeMonitor(G), StateMonitor(G, [v], record=[0, n - 1], when=when)]
    if name == "gap":
        G.set(v, 1.3 * rng.random(n))
        S = Synapses(G, G, summed={names["Igap"]: m.summed[names["Igap"]]}, name="s")
        i, j = np.repeat(np.arange(n), n), np.tile(np.arange(n), n)
        S.connect(i, j)
        S.set(names["w"], 6.0 / n * rng.random(n * n))
        syn = [S]
    else:
        G.set(v, synth.cuba_v0(3, n) if name == "cuba" else -0.06 + 0.05 * rng.random(n))
        syn = []
        for k, (a, b) in {"exc": (0, n * 4 // 5), "inh": (n * 4 // 5, n)}.items():
            S = Synapses(G[a:b], G, m.pathways[k], name=k)
            S.connect(*np.nonzero(rng.random((b - a, n)) < 0.1))
            syn.append(S)
    net = Network(G, *syn, *mons, dt=1e-4, **options)
    net.run(150)
    return net, [G.get(names.get(x, x)) for x in ("v",)] + [mons[0].i, mons[0].step, mons[1].values()]


@pytest.mark.parametrize("name, names, when, chip", [
    ("cuba", {"v": "s", "ge": "q", "gi": "step"}, "start", False),
    ("cobahh", {"m": "hi", "n": "w", "h": "x", "ge": "lane", "gi": "s", "v": "step"}, "end", True),
    ("gap", {"v": "x", "Igap": "u", "w": "lo"}, "start", True),
])
def test_awkward_names(name, names, when, chip):
    net, got = _group(700 if name == "cuba" else 100, name, names, when)
    own = {"Igap": "Igap", "w": "w"} if name == "gap" else {}
    _, want = _group(700 if name == "cuba" else 100, name, own, when, tile=256)
    assert net.in_launch is not None and (net.resident is None) == chip
    assert len(want[1]) > 0
    for x, y in zip(got, want):
        assert np.array_equal(x, y)


def test_awkward_names_of_targets():
    from brian2_amd import Network, NeuronGroup, SpikeGeneratorGroup, SpikeMonitor, Synapses

    out = []
    for names, options in (({"ge": "m", "v": "s", "w": "k", "Apre": "at", "Apost": "id"}, {}), ({}, {"tile": 256})):
        rng = np.random.default_rng(2)
        model = _model("stdp", names)
        step, idx = np.nonzero(rng.random((300, 200)) < 0.02)
        src = SpikeGeneratorGroup(200, idx, timebins=step)
        G = NeuronGroup(5, model, name="g")
        G.set(names.get("v", "v"), -0.06 + 0.006 * rng.random(5))
        S = Synapses(src, G, model.pathways["pre"], on_post=model.pathways["post"], name="s")
        S.connect(np.repeat(np.arange(200), 5), np.tile(np.arange(5), 200))
        S.set(names.get("w", "w"), 0.01 * rng.random(1000))
        mon = SpikeMonitor(G)
        net = Network(src, G, S, mon, dt=1e-4, **options)
        net.run(300)
        assert (net.resident is not None) == (not options)
        out.append([G.get(names.get("v", "v")), mon.i, mon.step] + [S.get(names.get(x, x)) for x in ("w", "Apre", "Apost")])
    assert len(out[1][1]) > 0
    for x, y in zip(*out):
        assert np.array_equal(x, y)


def _drawn(kind, seed, names=None):
    """A network of a seed's draw, and what a run leaves."""
    from brian2_amd import Model, Network, NeuronGroup, SpikeGeneratorGroup, SpikeMonitor, StateMonitor, Synapses, synth

    rng = np.random.default_rng(seed)
    if kind in ("cuba", "staged"):
        c = synth.cuba_network(N=700, seed=seed, network_options={"tile": 256} if kind == "staged" else {})
        net, G = c["net"], c["G"]
    elif kind == "cobahh":
        c = synth.cobahh_network(N=700, seed=seed)
        net, G = c["net"], c["G"]
    elif kind in ("fused", "separate"):
        c = synth.cuba_synw_network(N=6000, K=1000, seed=seed, network_options={"fuse": kind == "fused"})
        net, G = c["net"], c["G"]
    elif kind == "targets":
        m = Model.load("stdp")
        step, idx = np.nonzero(rng.random((100, 50)) < 0.1)
        src = SpikeGeneratorGroup(50, idx, timebins=step)
        G = NeuronGroup(3, m)
        G.v = -0.055
        S = Synapses(src, G, m.pathways["pre"], on_post=m.pathways["post"])
        S.connect(np.repeat(np.arange(50), 3), np.tile(np.arange(3), 50))
        S.set("w", 0.05 * rng.random(150))
        net = Network(src, G, S, SpikeMonitor(G), dt=1e-4)
    else:
        m = Model.load("gap")
        n = 60 if kind == "sums" else 1000
        G = NeuronGroup(n, m)
        G.v = 1.3 * rng.random(n)
        S = Synapses(G, G, summed={"Igap": m.summed["Igap"]})
        S.connect(rng.integers(0, n, 40 * n), np.repeat(np.arange(n), 40))
        S.set("w", rng.random(40 * n) / 40)
        net = Network(G, S, dt=1e-4, **({"tile": 128} if kind == "summed" else {}))
    net.run(150)
    return net, [G.get(v) for v in G.vars]


@pytest.mark.parametrize("kind", ["cuba", "staged", "cobahh", "fused", "separate", "targets", "sums", "own sum", "summed"])
def test_a_network_drawn_again_finds_its_kernels_compiled(kind):
    """Names that the package gives (neurongroup_3) and the draw of the synapses compile nothing
    anew, and the kernels found are the right ones."""
    from brian2_amd import runtime

    net, first = _drawn(kind, 1)
    modules = len(runtime.Device.get()._modules)
    for seed in (2, 3, 1):
        net, out = _drawn(kind, seed)
        assert len(runtime.Device.get()._modules) == modules, seed
    assert all(np.array_equal(x, y) for x, y in zip(first, out))


@pytest.mark.parametrize("kind, launches", [("cuba", ["step", "gather", "gather"]), ("cobahh", ["step", "gather", "gather"]),
                                            ("targets", ["step", "step", "gather"]), ("sums", ["step"])])
def test_profiles_of_networks_that_step_in_one_launch(kind, launches):
    """profile() times the code objects one by one, as for any network, and leaves what a run
    would: state, records, counts, and what a snapshot restores."""
    a, b = _drawn(kind, 5)[0], _drawn(kind, 5)[0]
    assert b.in_launch is not None

    def results(net):
        out = [g._dev[v].cpu().numpy() for g in net.groups for v in g.vars] + [net.n_events, net.t_step]
        out += [s.get(v) for s in net.paths for v in s.syn_vars]
        return out + [x for m in net.smons for x in (m.i, m.step, m.t_, m.count)]

    assert kind == "sums" or len(results(b)[-4]) > 0
    a.run(60)
    b.store()
    for _ in range(2):
        prof = b.profile(60)
        assert [k for k, _, _ in prof] == launches and all(ms > 0.0 for _, _, ms in prof)
        assert [n for _, n, _ in prof] == [o.name for o in list(b.groups) + list(b.paths)]
        assert all(np.array_equal(x, y) for x, y in zip(results(a), results(b)))
        b.restore()
    b.profile(60)
    a.run(40)
    b.run(40)
    assert b.in_launch is not None and all(np.array_equal(x, y) for x, y in zip(results(a), results(b)))
