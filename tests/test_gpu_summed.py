"""Summed variables on the device against Brian's cython runtime (golden_gap.npz:
examples/synapses/gapjunctions.py at 300 neurons, all-to-all, per-synapse weights)."""
import numpy as np
import pytest

import oracle_py as O

pytestmark = pytest.mark.gpu


def _gap_network(meta):
    from brian2_amd import Model, Network, NeuronGroup, SpikeMonitor, Synapses

    inp = O.gap_inputs(meta["seed"])
    m = Model.load("gap")
    G = NeuronGroup(meta["n"], m, name="neurons")
    G.v = inp["v"]
    S = Synapses(G, G, summed={"Igap": m.summed["Igap"]}, name="gap")
    S.connect(inp["pre"], inp["post"])
    S.set("w", inp["w"])
    mon = SpikeMonitor(G)
    return Network(G, S, mon, dt=meta["dt"]), G, mon


def test_gap_junctions_bitexact_vs_brian():
    z, meta = O.load_golden("gap")
    net, G, mon = _gap_network(meta)
    net.run(meta["n_steps"])
    assert len(mon.i) == len(z["i"])
    assert np.array_equal(mon.i, z["i"]) and np.array_equal(mon.step, z["step"])
    assert np.array_equal(np.stack([G.get("v"), G.get("Igap")]), z["final"])


def test_gap_junctions_in_pieces():
    z, meta = O.load_golden("gap")
    net, G, mon = _gap_network(meta)
    for k in (1, 999, 1000, 3000):
        net.run(k)
    assert np.array_equal(mon.i, z["i"]) and np.array_equal(mon.step, z["step"])
    assert np.array_equal(G.get("v"), z["final"][0])


@pytest.mark.parametrize("lanes", [1, 64])
@pytest.mark.parametrize("float_t", ["double", "float"])
def test_summed_fold_at_the_chunk_edges(lanes, float_t, monkeypatch):
    """One step of a summed variable over targets with 0 to 1100 synapses, around the edges
    of a wave's chunk: every sum equals the sequential fold in synapse order exactly."""
    from brian2_amd import Model, Network, NeuronGroup, Synapses
    from brian2_amd.kernels import SummedKernel

    monkeypatch.setattr(SummedKernel, "lanes_for", staticmethod(lambda n_syn, n_tgt: lanes))
    rng = np.random.default_rng(3)
    n = 41
    degree = np.array([0, 1, 2, 15, 16, 17, 63, 64, 65, 511, 512, 513, 527, 528, 1023, 1024, 1025, 1100])
    post = rng.permutation(np.repeat(np.arange(len(degree)) + 5, degree))
    pre = rng.integers(0, n, len(post))
    ft = np.float64 if float_t == "double" else np.float32
    v, w = (0.9 * rng.random(n)).astype(ft), rng.standard_normal(len(post))
    m = Model.load("gap")
    G = NeuronGroup(n, m, float_t=float_t)
    G.v = v
    S = Synapses(G, G, summed={"Igap": m.summed["Igap"]})
    S.connect(pre, post)
    S.set("w", w)
    Network(G, S, dt=1e-4).run(1)
    want = np.zeros(n, ft)
    for i, j, x in zip(pre, post, w):
        want[j] = want[j] + ft(x * np.float64(v[i] - v[j]))
    assert np.array_equal(G.get("Igap"), want)


@pytest.mark.parametrize("n, t, float_t, when", [(20, (0, 20), "double", "start"), (257, (3, 250), "float", "end"),
                                                 (301, (0, 301), "double", "end")])
def test_a_groups_own_sum_equals_two_launches(n, t, float_t, when):
    """A summed variable that the group forms in its own step: as with a launch of its own
    (tile given), over runs in pieces, restore, state set between runs and a change of dt."""
    from brian2_amd import Model, Network, NeuronGroup, PopulationRateMonitor, SpikeMonitor, StateMonitor, Synapses

    def run(**options):
        rng = np.random.default_rng(n)
        m = Model.load("gap")
        G = NeuronGroup(n, m, float_t=float_t)
        G.v = 1.3 * rng.random(n)  # some above the threshold
        S = Synapses(G, G[t[0]:t[1]], summed={"Igap": m.summed["Igap"]})
        i, j = np.nonzero((rng.random((n, t[1] - t[0])) < 0.95) & (np.arange(t[1] - t[0]) != 7))
        o = rng.permutation(len(i))
        S.connect(i[o], j[o])
        S.set("w", 6.0 / n * rng.random(len(i)))
        mons = [SpikeMonitor(G), StateMonitor(G, ["v", "Igap"], record=[0, 7, n - 1], when=when), PopulationRateMonitor(G)]
        net = Network(G, S, *mons, dt=1e-4, **options)
        net.run(3)
        net.run(150)
        net.store()
        net.run(1)
        net.restore()
        G.v = G.get("v")[::-1].copy()
        net.run(70)
        net.run(40, dt=5e-5)
        return G, [G.get("v"), G.get("Igap"), mons[0].i, mons[0].step, mons[1].values(), mons[2].count]

    G, got = run()
    H, want = run(tile=256)
    assert G.own_sum is not None and H.own_sum is None
    assert len(want[2]) > 0
    for x, y in zip(got, want):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("n, t, float_t, when", [(1, (0, 1), "double", "start"), (20, (0, 20), "float", "end"),
                                                 (257, (3, 250), "double", "end"), (384, (0, 384), "double", "start"),
                                                 (385, (0, 385), "double", "end"), (768, (0, 768), "float", "start")])
def test_own_sums_in_a_launch_and_launch_by_launch(n, t, float_t, when, monkeypatch):
    """All steps in a launch (up to 768 words, synapses in registers up to 512 a target), the group's
    own sum launch by launch and a launch for the sum: the same."""
    from brian2_amd import Model, Network, NeuronGroup, SpikeMonitor, StateMonitor, Synapses, chip
    from brian2_amd.kernels import SummedKernel

    monkeypatch.setattr(SummedKernel, "lanes_for", staticmethod(lambda n_syn, n_tgt: 64))

    def run(**options):
        rng = np.random.default_rng(n)
        m = Model.load("gap")
        G = NeuronGroup(n, m, float_t=float_t)
        G.v = 1.3 * rng.random(n)
        S = Synapses(G, G[t[0]:t[1]], summed={"Igap": m.summed["Igap"]})
        i, j = np.nonzero(rng.random((n, t[1] - t[0])) < 0.97)
        S.connect(i, j)
        S.set("w", 6.0 / n * rng.random(len(i)))
        mons = [SpikeMonitor(G), StateMonitor(G, ["v", "Igap"], record=sorted({0, n - 1}), when=when)]
        net = Network(G, S, *mons, dt=1e-4, **options)
        net.run(1)
        net.run(90)
        net.run(30, dt=5e-5)
        return net, [G.get("v"), G.get("Igap"), mons[0].i, mons[0].step, mons[1].values()]

    a, got = run()
    assert (a.in_launch is not None) == (n != 385)
    b, want = run(tile=256)
    assert b.in_launch is None
    monkeypatch.setattr(chip.SumSteps, "takes", classmethod(lambda *x: False))
    c, alone = run()
    assert c.in_launch is None and c.groups[0].own_sum is not None
    assert n == 1 or len(want[2]) > 0
    for x, y, z in zip(got, want, alone):
        assert np.array_equal(x, y) and np.array_equal(z, y)


@pytest.mark.parametrize("when", ["start", "end"])
@pytest.mark.parametrize("form", ["all steps in a launch", "its own step", "a wave per target", "a thread per target",
                                  "another group"])
def test_recorded_sums_are_those_of_the_monitors_point(form, when, monkeypatch):
    """A step forms the sums first.  A monitor at the step's start has the sum of the step before,
    one at its end the step's own: the sequential fold of the states recorded beside it, however
    the steps are cut into runs."""
    from brian2_amd import Model, Network, NeuronGroup, StateMonitor, Synapses, chip
    from brian2_amd.kernels import SummedKernel

    n = 70
    if form == "its own step":
        monkeypatch.setattr(chip.SumSteps, "takes", classmethod(lambda *x: False))
    if form == "a thread per target":
        monkeypatch.setattr(SummedKernel, "lanes_for", staticmethod(lambda *x: 1))
    rng = np.random.default_rng(9)
    pre, post = np.nonzero(rng.random((n, n - 5)) < 0.7)  # five neurons that are no targets
    v0, w = 1.3 * rng.random(n), 6.0 / n * rng.random(len(pre))
    rows = []
    for pieces in ((40,), (1, 19, 20)):
        m = Model.load("gap")
        H = NeuronGroup(n, m, name="h")
        H.v = v0
        H.Igap = 0.25
        G = H
        if form == "another group":
            G = NeuronGroup(n, Model.load("gap"), name="g")
            G.v = v0[::-1]
        S = Synapses(G, H[:n - 5], summed={"Igap": m.summed["Igap"]})
        S.connect(pre, post)
        S.set("w", w)
        mons = {x: StateMonitor(x, ["v", "Igap"], record=np.arange(n), when=when) for x in {G, H}}
        net = Network(*{G, H}, S, *mons.values(), dt=1e-4, **({"tile": 256} if form == "a wave per target" else {}))
        for k in pieces:
            net.run(k)
        assert (net.in_launch is not None) == (form == "all steps in a launch")
        assert (H.own_sum is not None) == (form in ("all steps in a launch", "its own step"))
        (vh, ih), vg = mons[H].values(), mons[G].values()[0]
        rows.append(ih)
        # the states that step s's sums read: recorded at its start, or at the end of step s - 1
        for s in range(39):
            want = np.full(n, 0.25)
            want[:n - 5] = 0.0
            for i, j, x in zip(pre, post, w):
                want[j] = want[j] + x * (vg[i, s] - vh[j, s])
            assert np.array_equal(ih[:, s + 1], want), s
        if when == "start":
            assert np.array_equal(ih[:, 0], np.full(n, 0.25))
    assert np.array_equal(*rows)


@pytest.mark.parametrize("n, own", [(300, True), (768, True), (769, False), (40001, False)])
def test_sums_that_read_nothing_of_their_sources(n, own):
    """The sum of a target's weights, say: as with a launch of its own, whatever the size."""
    from brian2_amd import Model, Network, NeuronGroup, Synapses

    out = []
    for options in ({}, {"tile": 256}):
        rng = np.random.default_rng(n)
        m = Model.load("gap")
        sp = m.summed["Igap"]
        sp.vector = [dict(sp.vector[0], expr="w")]
        G = NeuronGroup(n, m)
        G.v = 1.3 * rng.random(n)
        S = Synapses(G, G, summed={"Igap": sp})
        post = np.repeat(np.arange(n), 24)
        S.connect(rng.integers(0, n, len(post)), post)
        S.set("w", rng.random(len(post)) / 24)
        net = Network(G, S, dt=1e-4, **options)
        net.run(1)
        net.run(20)
        assert (net.in_launch is not None) == (own and not options)
        out.append([G.get("v"), G.get("Igap")])
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
