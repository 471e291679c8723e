"""The neuron and synapse kernels are compiled for what the populations and projections of a model have: few inputs and at most a constant current, the single-launch
step's, and everything a description can say; stored static rows, those and plastic ones, delayed ones, and all.  On either side of each line, against the CPU oracle bit for bit (weights are multiples of 2^-8 and inputs
keep nothing between steps, so every fp32 sum is exact in any order)."""
import numpy as np
import pytest

from genn_amd.netspec import CurrentSource, Net, Pop, Syn
from parity import run_side_by_side

pytestmark = pytest.mark.gpu

LIF = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, TauRefrac=3.0)


def _net(inputs, sources, kinds, steps=40, n_src=150, n_trg=333):
    rng = np.random.default_rng(inputs * 10 + len(sources))
    net = Net(name="instances", dt=1.0, steps=steps)
    for name, n, offset in (("S", n_src, 0.8), ("T", n_trg, 0.7)):
        net.pops.append(Pop(name, "lif", n, dict(LIF, Ioffset=offset), {"V": rng.uniform(-60.0, -50.0, n).astype(np.float32), "RefracTime": np.zeros(n, np.float32)}))
    for k in range(inputs):
        length, stride = rng.integers(0, 21, n_src).astype(np.uint32), 20
        ind = np.sort(np.stack([rng.choice(n_trg, stride, replace=False) for _ in range(n_src)]), axis=1)
        for r in range(n_src):
            ind[r, :length[r]] = np.sort(ind[r, :length[r]])
        kind = kinds[k % len(kinds)]
        syn = Syn(f"P{k}", "S", "T", wum="static" if kind == "axonal" else kind, axonal_delay_steps=2 if kind == "axonal" else 0, psm="deltacurr", row_stride=stride, row_length=length, ind=ind.astype(np.uint32),
                  g=(rng.integers(-40, 120, (n_src, stride)) / 256.0).astype(np.float32))
        if kind == "static_delay":
            syn.d, syn.max_den_delay = rng.integers(0, 3, (n_src, stride)).astype(np.uint8), 3
        net.syns.append(syn)
    for k, kind in enumerate(sources):
        noise = (rng.integers(-64, 64, (steps, n_trg)) / 256.0).astype(np.float32) if kind == "noise" else None
        net.css.append(CurrentSource(f"C{k}", kind, "T", amp=0.125 * (k + 1), noise=noise))
    return net


S, D = ("static",), ("static_delay",)


@pytest.mark.parametrize("inputs,sources,kinds", [(1, (), S), (4, ("dc",), S), (5, ("dc",), S), (8, (), S), (4, ("dc", "dc"), S), (2, ("noise",), S),
                                                  (1, (), D), (2, ("noise",), D), (3, ("dc",), D), (2, ("dc", "noise"), D), (8, (), D),
                                                  (2, (), S + D), (2, ("dc",), S + ("axonal",)), (2, (), S + ("static_reverse",)), (3, (), D + S + ("axonal",))])
def test_populations_and_projections_on_either_side_of_what_an_instance_has(inputs, sources, kinds):
    net = _net(inputs, sources, kinds)
    model, _, counts = run_side_by_side(net)
    model.unload()
    assert counts["S"] > 0 and counts["T"] > 0


@pytest.mark.parametrize("sources", [(), ("dc",), ("noise",)])
@pytest.mark.parametrize("kinds", [S, D, D + S])
def test_several_neurons_a_lane_with_delays_and_without(sources, kinds, monkeypatch):
    monkeypatch.setenv("GENNMI_NEURON_BULK", "1")
    model, _, counts = run_side_by_side(_net(2, sources, kinds, n_trg=1333))
    assert model.runner_info()["bulk_neuron_kernel"] and counts["T"] > 0
    model.unload()
