"""Targets of a spike generator through plastic synapses, a wave each
(brian2_amd/targets.py), against the staged launches (tile given), bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VARS = ("w", "Apre", "Apost", "lastupdate")


def _run(n, m, p, per_step, float_t, some=False, **options):
    from brian2_amd import Model, Network, NeuronGroup, SpikeGeneratorGroup, SpikeMonitor, Synapses

    rng = np.random.default_rng(n + m)
    idx, step = [], []
    for s, k in per_step(n):
        idx.append(rng.permutation(n)[:k])
        step.append(np.full(k, s))
    src = SpikeGeneratorGroup(n, np.concatenate(idx), timebins=np.concatenate(step))
    model = Model.load("stdp")
    G = NeuronGroup(m, model, float_t=float_t, name="g")
    G.v = -0.06 + 0.006 * rng.random(m)
    a = src[n // 5:n - n // 7] if some else src
    S = Synapses(a, G, model.pathways["pre"], on_post=model.pathways["post"], name="s")
    i, j = np.nonzero((rng.random((a.N, m)) < p) & (np.arange(m) != m // 2))  # a target without synapses
    o = rng.permutation(len(i))
    S.connect(i[o], j[o])
    S.set("w", 0.01 * rng.random(len(i)) * min(1.0, 500.0 / n))
    mon = SpikeMonitor(G[m // 4:])
    net = Network(src, G, S, mon, dt=1e-4, **options)
    for k in (1, 150, 49):
        net.run(k)
    net.store()
    net.run(30)
    net.restore()
    net.run(100)
    return net, [S.get(v) for v in VARS] + [G.get(v) for v in G.vars] + [
        mon.i, mon.step, mon.count, np.array([net.n_events])]


def _steady(n):  # gaps, and a volley of all sources
    return [(s, (s * 7) % 5) for s in range(3, 280) if s % 4] + [(281, n)] + [(290, 1)]


def _full_batches(n):  # every step 64 entries
    return [(s, min(64, n)) for s in range(0, 60)]


def _over(n):  # beyond a batch, off its bounds
    return [(s, min(65 + s, n)) for s in range(0, 300, 2)]


@pytest.mark.parametrize("n, m, p, per_step, float_t, some", [
    (1000, 20, 1.0, _steady, "double", False),
    (64, 3, 1.0, _full_batches, "double", False),
    (200, 5, 0.4, _over, "float", True),
    (333, 2, 0.7, _steady, "double", True),
    (4000, 9, 1.0, _over, "double", False),
])
def test_targets_equal_the_staged_launches(n, m, p, per_step, float_t, some):
    a, got = _run(n, m, p, per_step, float_t, some)
    b, want = _run(n, m, p, per_step, float_t, some, tile=256)
    assert a.resident is not None and b.resident is None
    assert want[-1][0] > 0 and want[1].max() > 0
    for x, y in zip(got, want):
        assert np.array_equal(x, y)


def test_networks_that_are_not_taken():
    """A second synapse of a pair and synapses beyond the LDS keep the staged launches."""
    from brian2_amd import Model, Network, NeuronGroup, SpikeGeneratorGroup, Synapses

    model = Model.load("stdp")
    for n, twice in ((10, True), (6000, False)):
        src = SpikeGeneratorGroup(n, [0, 1], timebins=[1, 2])
        G = NeuronGroup(2, model)
        S = Synapses(src, G, model.pathways["pre"], on_post=model.pathways["post"])
        i, j = np.repeat(np.arange(n), 2), np.tile(np.arange(2), n)
        S.connect(np.append(i, i[:1]), np.append(j, j[:1])) if twice else S.connect(i, j)
        net = Network(src, G, S, dt=1e-4)
        net.run(5)
        assert net.resident is None
