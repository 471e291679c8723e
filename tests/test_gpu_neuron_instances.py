"""The neuron and synapse kernels are compiled for what the populations and projections of a model have: few inputs and at most a constant current, the single-launch
step's, and everything a description can say; stored static rows, those and plastic ones, delayed ones, and all.  On either side of each line, against the CPU oracle bit for bit (weights are multiples of 2^-8 and inputs
keep nothing between steps, so every fp32 sum is exact in any order)."""
import copy

import numpy as np
import pytest

from genn_amd.genn_model import model_from_net
from genn_amd.netspec import CurrentSource, Net, Pop, Syn
from oracle.genn_cpu import OracleNet
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


@pytest.mark.parametrize("inputs,sources,kinds,neurons,synapses", [
    (1, (), S, True, True), (4, ("dc",), S, True, True), (5, ("dc",), S, False, True), (8, (), S, False, True), (4, ("dc", "dc"), S, False, True), (2, ("noise",), S, False, True),
    (1, (), D, True, True), (2, ("noise",), D, True, True), (2, ("poisson_exp",), D, True, True), (2, (), S + D, False, False), (2, ("dc",), S + ("axonal",), False, False),
    (2, (), S + ("static_reverse",), False, False)])
def test_which_instances_a_network_runs(inputs, sources, kinds, neurons, synapses):
    """The instances that the tests above and below mean to run are those that a network is given."""
    net = _net(inputs, tuple(k for k in sources if k != "poisson_exp"), kinds)
    if "poisson_exp" in sources:
        net.css.append(CurrentSource("C", "poisson_exp", "T", params=dict(weight=0.125, tauSyn=0.5, rate=800.0)))
    model = model_from_net(net)
    model.load(num_recording_timesteps=1)
    info = model.runner_info()
    assert info["single_launch_step"] == (kinds == D) and (info["combined_synapse_launch"] or not synapses or kinds == D)
    assert (info["lean_neuron_kernel"], info["narrow_synapse_kernel"]) == (neurons, synapses)
    model.unload()


@pytest.mark.parametrize("rule", ["stdp_trace", "stdp_additive"])
@pytest.mark.parametrize("kinds,synapses", [((), True), (S, True), (D, False), (("static_reverse",), False), (S + D, False)])
def test_learning_projections_alone_and_beside_others(kinds, synapses, rule):
    """Time constants so long that traces do not decay: every change of a weight is a multiple of 2^-8, so that sums are exact in any order here too."""
    net = _net(1 + len(kinds), ("dc",), S + kinds)
    plastic = net.syns[0]
    plastic.wum, plastic.wum_params = rule, dict(tauPlus=1e30, tauMinus=1e30, aPlus=3.0 / 256.0, aMinus=2.0 / 256.0, wMin=-0.25, wMax=0.5)
    model, _, counts = run_side_by_side(net)
    assert counts["S"] > 0 and counts["T"] > 0
    valid = np.arange(plastic.ind.shape[1])[None, :] < plastic.row_length[:, None]
    assert (model.synapse_populations["P0"].vars["g"].pull_from_device().reshape(valid.shape)[valid] != plastic.g[valid]).mean() > 0.5
    info = model.runner_info()
    assert info["postsyn_blocks"] > 0 and info["narrow_synapse_kernel"] == synapses and (info["postsynaptic_in_combined_launch"] or not synapses)
    model.unload()


@pytest.mark.parametrize("n_src,n_trg", [(1, 255), (257, 513), (700, 63)])
def test_batches_of_spike_sources_and_few_inputs(n_src, n_trg):
    """Lanes beyond a population and beyond a batch's share of it; every batch is the oracle's run of that batch's spikes."""
    batches, steps, gen = 3, 40, np.random.default_rng(n_src)
    net = _net(2, ("dc",), S, steps=steps, n_src=max(n_src, 20), n_trg=n_trg)
    net.pops[0] = Pop("S", "ssa", n_src, {}, {})
    for syn in net.syns:
        syn.row_length, syn.ind, syn.g = syn.row_length[:n_src], syn.ind[:n_src], syn.g[:n_src]
    fire = gen.random((batches, n_src, steps)) < 0.1
    counts = fire.sum(axis=2).reshape(-1)
    end = np.cumsum(counts).astype(np.uint32).reshape(batches, n_src)
    times = np.nonzero(fire)[2].astype(np.float32)
    oracles = []
    for b in range(batches):
        one = copy.deepcopy(net)
        own = np.nonzero(fire[b])[1].astype(np.float32)
        own_end = np.cumsum(fire[b].sum(axis=1)).astype(np.uint32)
        one.pops[0].vars, one.pops[0].spike_times = {"startSpike": (own_end - fire[b].sum(axis=1)).astype(np.uint32), "endSpike": own_end}, own
        oracles.append(OracleNet(one))
    net.pops[0].vars, net.pops[0].spike_times = {"startSpike": (end.reshape(-1) - counts).astype(np.uint32).reshape(batches, n_src), "endSpike": end}, times
    model = model_from_net(net, batch_size=batches)
    model.load(num_recording_timesteps=steps)
    info = model.runner_info()
    assert info["lean_neuron_kernel"] and info["narrow_synapse_kernel"] and not info["bulk_neuron_kernel"]
    spikes = 0
    for step in range(steps):
        model.step_time()
        got = {name: model.neuron_populations[name].current_spikes for name in "ST"}
        for b, oracle in enumerate(oracles):
            oracle.step()
            for name in "ST":
                assert np.array_equal(got[name][b], oracle.spikes(name)), (step, b, name)
                spikes += len(oracle.spikes(name))
    assert spikes > 0
    v = model.neuron_populations["T"].vars["V"].pull_from_device().reshape(batches, -1)
    for b, oracle in enumerate(oracles):
        assert np.array_equal(v[b], oracle.var("T", 0))
    model.unload()


@pytest.mark.parametrize("inputs,sources", [(3, ()), (2, ("dc", "noise")), (1, ("dc", "dc")), (8, ("noise",))])
def test_single_launch_steps_of_more_inputs_or_sources(inputs, sources):
    """What the lean neuron instance of the single-launch step does not take runs beside the synapse code for everything: the instance for delayed rows
    alone made such a step up to 8 % longer."""
    model, _, counts = run_side_by_side(_net(inputs, sources, D))
    info = model.runner_info()
    assert info["single_launch_step"] and not info["lean_neuron_kernel"] and not info["narrow_synapse_kernel"]
    assert counts["S"] > 0 and counts["T"] > 0
    model.unload()
