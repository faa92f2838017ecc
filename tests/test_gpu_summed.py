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
