"""The neuron update for large populations (four neurons per lane, all inputs requested before anything is stored),
forced onto small networks: it must leave every array exactly as the one-neuron-per-lane kernel and the CPU oracle do."""
import numpy as np
import pytest

from genn_amd import configs, rng
from genn_amd.netspec import Net, Pop, Syn
from parity import run_side_by_side

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _bulk(monkeypatch):
    monkeypatch.setenv("GENNMI_NEURON_BULK", "1")
    monkeypatch.setenv("GENNMI_RESIDENT", "0")


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 5000])
def test_ragged_population_sizes(n, monkeypatch):
    """Sizes around the chunk (64), the wave's share (256) and the work-group's share (1024); everyone fires in step 0."""
    monkeypatch.setenv("GENNMI_TILE_FLOATS", "0")
    lif = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=1.0, TauRefrac=2.0)
    net = Net(name="ragged_bulk", dt=1.0, steps=40)
    net.pops.append(Pop("A", "lif", n, dict(lif), {"V": np.full(n, -50.5, np.float32), "RefracTime": np.zeros(n, np.float32)}))
    m = max(1, n // 2)
    net.pops.append(Pop("B", "lif", m, dict(lif, Ioffset=0.2), {"V": np.full(m, -60.0, np.float32), "RefracTime": np.zeros(m, np.float32)}))
    stride = 5
    row_length = (rng.randint(3, 1, 0, n, stride + 1)).astype(np.uint32)
    ind = np.sort(rng.randint(3, 2, 0, n * stride, m).reshape(n, stride), axis=1).astype(np.uint32)
    net.syns.append(Syn("AB", "A", "B", wum="static", psm="expcurr", tau=5.0, row_stride=stride, row_length=row_length, ind=ind,
                        g=np.full((n, stride), 1.5, np.float32)))
    model, oracle, counts = run_side_by_side(net, check_every=10, exact=True)
    assert model.runner_info()["bulk_neuron_kernel"]
    assert counts["A"] >= n
    model.unload()


def test_balanced_network_two_postsynaptic_models():
    net = configs.vogels_abbott(n=4000, steps=600)
    model, oracle, counts = run_side_by_side(net, check_every=100, exact=True)
    assert model.runner_info()["bulk_neuron_kernel"]
    assert counts["E"] > 500 and counts["I"] > 100
    model.unload()


def test_many_work_groups_every_one_with_spikes():
    """70,000 uncoupled-looking neurons with staggered phases: 69 work-groups, so queue offsets cross the boundary between
    two groups of 64 whose totals are published separately, and nearly every work-group emits spikes in every step."""
    n = 70000
    lif = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=1.2, TauRefrac=1.0)
    net = Net(name="many_groups", dt=1.0, steps=40)
    net.pops.append(Pop("A", "lif", n, dict(lif), {"V": (-60.0 + 10.0 * rng.uniform(8, 1, 0, n)).astype(np.float32), "RefracTime": np.zeros(n, np.float32)}))
    net.pops.append(Pop("B", "lif", 300, dict(lif, Ioffset=0.1), {"V": np.full(300, -60.0, np.float32), "RefracTime": np.zeros(300, np.float32)}))
    ind = rng.randint(8, 2, 0, n, 300).reshape(n, 1).astype(np.uint32)
    net.syns.append(Syn("AB", "A", "B", wum="static", psm="expcurr", tau=5.0, row_stride=1, row_length=np.ones(n, np.uint32), ind=ind,
                        g=np.full((n, 1), 0.0078125, np.float32)))
    model, oracle, counts = run_side_by_side(net, check_every=10, exact=True)
    assert model.runner_info()["bulk_neuron_kernel"]
    assert counts["A"] > 3 * n
    model.unload()


def test_dendritic_delay_rings(monkeypatch):
    """Front slot of the delay ring read and cleared by the bulk kernel (microcircuit shape, fused postsynaptic models)."""
    net = configs.potjans(neuron_scale=0.05, connectivity_scale=1.0, steps=300)
    model, oracle, counts = run_side_by_side(net, check_every=50, exact=False, exact_steps=300)
    info = model.runner_info()
    assert info["bulk_neuron_kernel"] and not info["single_launch_step"]
    assert sum(counts.values()) > 100
    model.unload()


def test_izhikevich_with_noise_source():
    net = configs.izhikevich_fanout(n=6000, fanout=100, steps=150)
    model, oracle, counts = run_side_by_side(net, check_every=25, exact=False, exact_steps=60)
    assert model.runner_info()["bulk_neuron_kernel"]
    assert counts["N"] > 100
    model.unload()


def test_spike_sources_and_batches():
    """Convolution layer: spike-source chunks, LIF chunks and three batches through the bulk kernel; batch b must equal a
    batch-1 oracle run fed batch b's spike trains."""
    import copy
    from genn_amd.genn_model import model_from_net
    from oracle.genn_cpu import OracleNet
    B = 3
    nets = [configs.conv_toeplitz(h=12, w=12, ic=3, oc=5, steps=60, w_sd=0.6, batch_index=b) for b in range(B)]
    for net in nets:
        net.pop("Out").params["Ioffset"] = 0.4
    times = np.concatenate([n.pop("In").spike_times for n in nets])
    offs = np.cumsum([0] + [len(n.pop("In").spike_times) for n in nets])
    start = np.stack([n.pop("In").vars["startSpike"] + offs[b] for b, n in enumerate(nets)]).astype(np.uint32)
    end = np.stack([n.pop("In").vars["endSpike"] + offs[b] for b, n in enumerate(nets)]).astype(np.uint32)
    batched = copy.deepcopy(nets[0])
    batched.pop("In").vars = {"startSpike": start, "endSpike": end}
    batched.pop("In").spike_times = times
    model = model_from_net(batched, batch_size=B)
    model.load(num_recording_timesteps=60)
    assert model.runner_info()["bulk_neuron_kernel"]
    oracles = [OracleNet(n) for n in nets]
    total = 0
    for step in range(60):
        model.step_time()
        got = {name: model.neuron_populations[name].current_spikes for name in ("In", "Out")}
        for b, o in enumerate(oracles):
            o.step()
            for name in ("In", "Out"):
                assert np.array_equal(got[name][b], o.spikes(name)), f"step {step} batch {b}: {name} spikes differ"
                total += len(o.spikes(name))
    assert total > 500
    v = model.neuron_populations["Out"].vars["V"].pull_from_device().reshape(B, -1)
    for b, o in enumerate(oracles):
        np.testing.assert_allclose(v[b], o.var("Out", 0), rtol=1e-5)
    model.unload()


@pytest.mark.parametrize("per_lane", [2, 4, 8])
@pytest.mark.parametrize("n", [1, 63, 65, 1025, 4100])
def test_spike_sources_several_a_lane(n, per_lane, monkeypatch):
    """Sources that never fire, fire once, at the end of the spike times, and in every step; sizes around a chunk, a wavefront's and a work-group's share."""
    monkeypatch.setenv("GENNMI_NEURON_BULK", str(per_lane))
    steps, gen = 30, np.random.default_rng(n)
    fire = gen.random((n, steps)) < gen.choice([0.0, 0.03, 0.3, 1.0], (n, 1), p=[0.4, 0.3, 0.2, 0.1])
    fire[-1] = [k % 7 == 0 for k in range(steps)]
    end = np.cumsum(fire.sum(axis=1)).astype(np.uint32)
    lif = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=0.45, TauRefrac=2.0)
    net = Net(name="bulk_sources", dt=1.0, steps=steps)
    net.pops.append(Pop("S", "ssa", n, {}, {"startSpike": (end - fire.sum(axis=1)).astype(np.uint32), "endSpike": end}, spike_times=np.nonzero(fire)[1].astype(np.float32)))
    net.pops.append(Pop("T", "lif", 700, dict(lif), {"V": (-60.0 + 10.0 * rng.uniform(8, 1, 0, 700)).astype(np.float32), "RefracTime": np.zeros(700, np.float32)}))
    ind = np.sort(gen.integers(0, 700, (n, 4)), axis=1).astype(np.uint32)
    net.syns.append(Syn("ST", "S", "T", wum="static", psm="deltacurr", row_stride=4, row_length=np.full(n, 4, np.uint32), ind=ind, g=np.full((n, 4), 0.0625, np.float32)))
    model, oracle, counts = run_side_by_side(net, exact=True)
    assert model.runner_info()["bulk_neuron_kernel"] and counts["S"] == fire.sum()
    model.unload()


def test_chunks_of_spike_sources_do_not_wait_for_one_another(monkeypatch):
    """A layer's neurons and its 10^6 sources, eight chunks a lane, most with a spike: looked up one chunk after the other, a
    launch took 1.39 times as long as with four chunks a lane (21.9 us, 15.8), now 1.13 times (16.4, 14.5)."""
    from genn_amd.genn_model import GeNNModel, init_postsynaptic, init_toeplitz_connectivity, init_weight_update
    h, ic, oc, batch, steps, took = 64, 16, 32, 16, 24, {}
    n = h * h * ic
    fire = np.random.default_rng(5).random((batch * n, steps), np.float32) < 0.025
    end, times = np.cumsum(fire.sum(axis=1)).astype(np.uint32), np.nonzero(fire)[1].astype(np.float32)
    monkeypatch.setenv("GENNMI_CONV_STEP", "0")
    for per_lane in (4, 8):
        monkeypatch.setenv("GENNMI_NEURON_BULK", str(per_lane))
        model = GeNNModel("float", "sources", dt=1.0, batch_size=batch)
        model.timing_enabled = True
        src = model.add_neuron_population("S", n, "SpikeSourceArray", {}, {"startSpike": (end - fire.sum(axis=1)).astype(np.uint32).reshape(batch, n), "endSpike": end.reshape(batch, n)})
        src.set_extra_global_param("spikeTimes", times)
        trg = model.add_neuron_population("T", h * h * oc, "LIF", dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=0.3, TauRefrac=2.0), {"V": -60.0, "RefracTime": 0.0})
        shape = dict(conv_kh=3, conv_kw=3, conv_ih=h, conv_iw=h, conv_ic=ic, conv_oh=h, conv_ow=h, conv_oc=oc)
        model.add_synapse_population("ST", "TOEPLITZ", src, trg, init_weight_update("StaticPulse", {}, {"g": np.full((3, 3, ic, oc), 0.01, np.float32)}), init_postsynaptic("ExpCurr", {"tau": 5.0}),
                                     init_toeplitz_connectivity("Conv2D", shape))
        model.build()
        model.load()
        rounds = []
        for _ in range(steps - 4):
            before = model.neuron_update_time
            model.step_time()
            rounds.append(model.neuron_update_time - before)
        took[per_lane] = float(np.median(rounds))
        assert model.runner_info()["bulk_neuron_kernel"] and not model.runner_info()["conv_step_in_one_launch"]
        model.unload()
    assert 0.0 < took[8] < 1.25 * took[4], took
