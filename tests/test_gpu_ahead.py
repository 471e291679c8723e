"""run() on feed-forward layers: up to 128 steps at once, the layer's input over the steps as a matrix product on the matrix
cores.  Weights are multiples of 2^-8 and the postsynaptic model keeps nothing between steps (unless said otherwise), so every
fp32 sum is exact in any order and queues, rasters, state and event counts must be those of the CPU oracle bit for bit."""
import copy

import numpy as np
import pytest

from genn_amd import _abi, configs
from genn_amd.genn_model import model_from_net
from oracle.genn_cpu import OracleNet
from parity import compare_state

pytestmark = pytest.mark.gpu


def _net(kind, shape, steps, psm="deltacurr", batch_index=0):
    if kind == "dense":
        n_in, n_out = shape
        net = configs.dense_layer(n_in=n_in, n_out=n_out, rate_hz=120.0, steps=steps, w_sd=6.0 / np.sqrt(n_in))
        if batch_index:
            source = net.pop("In")
            source.vars["startSpike"], source.vars["endSpike"], source.spike_times = configs.poisson_spike_source(17, 50 + batch_index, n_in, 120.0, steps, 1.0)
    else:
        h, w, ic, oc, k = shape
        net = configs.conv_toeplitz(h=h, w=w, ic=ic, oc=oc, k=k, steps=steps, w_sd=3.0 / k, max_rate=200.0, ioffset=0.3, batch_index=batch_index)
    syn = net.syns[0]
    syn.g = (np.rint(syn.g * 256.0) / 256.0).astype(np.float32)
    syn.psm = psm
    return net


def _same_rasters(net, model, oracle, steps):
    model.pull_recording_buffers_from_device()
    for p in net.pops:
        words = (p.n + 31) // 32
        assert np.array_equal(model.neuron_populations[p.name].vars["recordSpk"].view.reshape(steps, words), oracle.record(p.name, steps).reshape(steps, words)), p.name
        assert np.array_equal(model.neuron_populations[p.name].current_spikes[0], oracle.spikes(p.name)), p.name


# sizes around a product's 32 columns, a chunk of 64 sources, a work-group's 512; output pixels around the four of a wavefront, channel
# counts that make an odd number of taps, more than 32 output channels, an even kernel
SHAPES = [("dense", (1, 1)), ("dense", (63, 31)), ("dense", (65, 33)), ("dense", (512, 64)), ("dense", (1300, 70)), ("dense", (300, 1000)), ("dense", (900, 40)),
          ("conv", (1, 1, 1, 1, 3)), ("conv", (5, 7, 3, 4, 3)), ("conv", (9, 6, 1, 33, 5)), ("conv", (8, 8, 16, 32, 3)), ("conv", (6, 5, 2, 40, 1))]


@pytest.mark.parametrize("kind,shape", SHAPES, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_runs_of_every_length_mixed_with_single_steps(kind, shape):
    """Runs on either side of the shortest that is taken at once, of a word of 32 steps and of the longest launch of 128."""
    chunks = [1, 7, 8, 1, 31, 32, 33, 2, 137, 0, 64]
    steps = sum(chunks)
    net = _net(kind, shape, steps)
    model = model_from_net(net)
    model.load(num_recording_timesteps=steps)
    assert model.runner_info()["feed_forward_ahead"]
    oracle = OracleNet(net, num_recording_timesteps=steps)
    for chunk in chunks:
        if chunk == 1:
            model.step_time()
        else:
            model.run(chunk)
        oracle.run(chunk)
        compare_state(net, model, oracle, f"after {chunk} more steps", exact=True)
    _same_rasters(net, model, oracle, steps)
    assert model.synaptic_event_count == oracle.events()
    assert int(np.unpackbits(oracle.record("In", steps).view(np.uint8)).sum()) > 0
    model.unload()


@pytest.mark.parametrize("kind,shape,model_name", [("dense", (700, 130), "izh"), ("dense", (700, 130), "lif"), ("conv", (9, 10, 3, 8, 3), "izh"), ("conv", (9, 10, 3, 8, 3), "lif")])
def test_exponential_synapses_and_both_neuron_models(kind, shape, model_name):
    """outPost carries over from step to step: the layer's sum is added to it at once instead of weight by weight.  LIF neurons contract
    such a difference: 1e-5.  The half steps of an Izhikevich neuron multiply one of V by 1 + (0.04 V + 2.5): 1.9^2 a step at -40 mV,
    2.5^2 at -25, 3.9^2 at +10, about 300 over the upstroke of a spike, and U keeps a share of it: 300 times three roundings of 2^-24
    is 5e-5 a spike, and the neurons fire fewer than ten times: 5e-4.  The rasters have to be identical."""
    steps = 100
    net = _net(kind, shape, steps, psm="expcurr")
    if model_name == "izh":
        out = net.pop("Out")
        out.model, out.params = "izh", dict(a=0.02, b=0.2, c=-65.0, d=8.0)
        out.vars = {"V": np.full(out.n, -65.0, np.float32), "U": np.full(out.n, -13.0, np.float32)}
    model = model_from_net(net)
    model.load(num_recording_timesteps=steps)
    assert model.runner_info()["feed_forward_ahead"]
    oracle = OracleNet(net, num_recording_timesteps=steps)
    model.run(steps)
    oracle.run(steps)
    if model_name == "lif":
        compare_state(net, model, oracle, "after the run", exact=False)
    else:
        for k, name in enumerate(("V", "U")):
            want = oracle.var("Out", k)
            assert np.abs(model.neuron_populations["Out"].vars[name].pull_from_device() - want).max() <= 5e-4 * np.abs(want).max(), name
    _same_rasters(net, model, oracle, steps)
    model.unload()


@pytest.mark.parametrize("kind,shape,batch", [("dense", (150, 70), 3), ("dense", (150, 70), 9), ("conv", (7, 6, 2, 5, 3), 3)])
def test_batches_recording_rows_reused_and_source_rewritten(kind, shape, batch, monkeypatch):
    """Batches are independent; a recording buffer of fewer rows than the run keeps the last step of each row; spike times and a queue
    written between runs count.  Against the same network stepped launch by launch."""
    steps, rows = 70, 6
    nets = [_net(kind, shape, steps, batch_index=b) for b in range(batch)]
    times = np.concatenate([n.pop("In").spike_times for n in nets])
    offs = np.cumsum([0] + [len(n.pop("In").spike_times) for n in nets])
    net = copy.deepcopy(nets[0])
    net.pop("In").vars = {v: np.stack([n.pop("In").vars[v] + offs[b] for b, n in enumerate(nets)]).astype(np.uint32) for v in ("startSpike", "endSpike")}
    net.pop("In").spike_times = times
    models = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        model = model_from_net(net, batch_size=batch)
        model.load(num_recording_timesteps=rows)
        assert model.runner_info()["feed_forward_ahead"] == (ahead == "1")
        models.append(model)
    start = models[0].neuron_populations["In"].vars["startSpike"].view.copy()
    for turn in range(2):
        for model in models:
            model.run(steps)
            model.pull_recording_buffers_from_device()
        for p in net.pops:
            a, b = (m.neuron_populations[p.name] for m in models)
            assert np.array_equal(a.vars["recordSpk"].view, b.vars["recordSpk"].view), p.name
            for name in ("V", "RefracTime", "startSpike"):
                if name in a.vars:
                    assert np.array_equal(a.vars[name].pull_from_device(), b.vars[name].pull_from_device()), name
            for k in range(batch):
                assert np.array_equal(a.current_spikes[k], b.current_spikes[k])
        assert models[0].synaptic_event_count == models[1].synaptic_event_count > 0
        for model in models:
            # the trains once more, 70 steps later, behind a queue of two spikes
            source = model.neuron_populations["In"]
            source.vars["spikeTimes"].view[:len(times)] = times + steps
            source.vars["startSpike"].view[:] = start
            source.vars["spkCnt"].view[:] = 2
            source.vars["spk"].view.reshape(batch, -1)[:, :2] = [3, 11]
            for v in ("spikeTimes", "startSpike", "spkCnt", "spk"):
                source.vars[v].push_to_device()
    for model in models:
        model.unload()


@pytest.mark.parametrize("kind,shape", [("dense", (200, 40)), ("conv", (6, 7, 2, 5, 3))])
def test_weights_that_are_not_finite_reach_their_own_spikes_only(kind, shape, monkeypatch):
    """0 * inf is NaN: an infinite weight of a source that is silent in a step must not touch that step."""
    steps = 40
    net = _net(kind, shape, steps)
    g = net.syns[0].g.reshape(-1)
    g[[5, 17]] = [np.inf, -np.inf]
    vs = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        monkeypatch.setenv("GENNMI_CONV_MFMA", ahead)       # (compared with the event-driven kernels: spike by spike)
        model = model_from_net(net)
        model.load(num_recording_timesteps=steps)
        assert model.runner_info()["feed_forward_ahead"] == (ahead == "1")
        model.run(steps)
        model.pull_recording_buffers_from_device()
        vs.append((model.neuron_populations["Out"].vars["V"].pull_from_device().copy(), model.neuron_populations["Out"].vars["recordSpk"].view.copy()))
        model.unload()
    assert np.array_equal(vs[0][0], vs[1][0], equal_nan=True) and np.array_equal(vs[0][1], vs[1][1])
    assert np.isfinite(vs[0][0]).any()


@pytest.mark.parametrize("kind,shape", [("dense", (200, 40)), ("conv", (6, 7, 2, 5, 3))])
def test_weights_too_small_to_split(kind, shape, monkeypatch):
    """Weights are split into three numbers of 8 bits for the matrix cores; below 2^-90 the lowest would underflow.  All weights are multiples
    of 2^-107 here: a step's sum is exact, and outPost differs by its rounding in each of forty steps, of a sum of at most four times the
    largest value left."""
    steps = 40
    net = _net(kind, shape, steps, psm="expcurr")
    syn = net.syns[0]
    syn.g = (syn.g * np.float32(2.0 ** -99)).astype(np.float32)
    got = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        monkeypatch.setenv("GENNMI_CONV_MFMA", ahead)
        model = model_from_net(net)
        model.load(num_recording_timesteps=steps)
        assert model.runner_info()["feed_forward_ahead"] == (ahead == "1")
        model.run(steps)
        got.append(model.synapse_populations[syn.name].vars["outPost"].pull_from_device().astype(np.float64).copy())
        model.unload()
    assert np.abs(got[1]).max() > 0.0
    assert np.abs(got[0] - got[1]).max() <= steps * 2.0 ** -24 * 4.0 * np.abs(got[1]).max()


def test_a_written_queue_that_names_a_neuron_twice(monkeypatch):
    """The DENSE kernel of a single step walks the queue as it is: so does the first step of a run."""
    steps = 20
    net = _net("dense", (90, 40), steps)
    got = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        model = model_from_net(net)
        model.load(num_recording_timesteps=steps)
        source = model.neuron_populations["In"]
        source.vars["spk"].view[:3] = [7, 7, 60]
        source.vars["spkCnt"].view[:] = 3
        for v in ("spk", "spkCnt"):
            source.vars[v].push_to_device()
        model.run(steps)
        got.append((model.neuron_populations["Out"].vars["V"].pull_from_device().copy(), model.synaptic_event_count))
        model.unload()
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]


# few and many inputs a pixel (one round of 64, seven), an odd number of them, more LDS than 64 KiB, channels beyond a product's 32
@pytest.mark.parametrize("shape,rate", [((8, 8, 16, 32, 3), 400.0), ((6, 9, 16, 8, 5), 250.0), ((4, 9, 17, 3, 5), 100.0), ((5, 7, 8, 33, 3), 300.0), ((5, 7, 3, 40, 3), 1000.0), ((9, 4, 13, 5, 2), 400.0)])
def test_convolutions_sum_to_the_same_bits_at_once_and_step_by_step(shape, rate, monkeypatch):
    """Weights of full precision: which inputs share a product must not change a bit.  (At these rates every step with spikes is one for the
    matrix cores when taken by itself; a kernel that its step kernel has no LDS for has weights whose sums are exact in any order.)"""
    h, w, ic, oc, k = shape
    steps = 41
    net = configs.conv_toeplitz(h=h, w=w, ic=ic, oc=oc, k=k, steps=steps, w_sd=1.0 / k, max_rate=rate, ioffset=0.3)
    exact = k * k * ic >= 400
    if exact:
        net.syns[0].g = (np.rint(net.syns[0].g * 256.0) / 256.0).astype(np.float32)
        net.syns[0].psm = "deltacurr"
    states = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        model = model_from_net(net)
        model.load(num_recording_timesteps=steps)
        assert model.runner_info()["feed_forward_ahead"] == (ahead == "1") and (exact or model.runner_info()["conv_on_matrix_cores"])
        model.run(steps)
        model.pull_recording_buffers_from_device()
        out, layer = model.neuron_populations["Out"], list(model.synapse_populations.values())[0]
        states.append([out.vars["recordSpk"].view.copy(), out.vars["V"].pull_from_device().copy(), layer.vars["outPost"].pull_from_device().copy(), model.synaptic_event_count])
        model.unload()
    assert states[0][3] == states[1][3] > 0 and np.any(states[0][0])
    for a, b in zip(states[0][:3], states[1][:3]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


# one spike and none, exactly four (the times a lane asks for at once) and one more, as many as steps; the step's length as a float and not, counts of
# steps that floats hold exactly, that they round to even ones, and beyond 32 bits
@pytest.mark.parametrize("dt,first_step", [(1.0, 0), (0.1, 3), (0.1, 1 << 22), (0.7, (1 << 24) + 5), (1.0, (1 << 25) + 1), (1.0, (1 << 32) - 40)])
def test_spike_times_off_the_grid_of_steps(dt, first_step, monkeypatch):
    """Times between steps, on them, next to them, several in one step (each is emitted a step later than the one before), in the past, not a number and
    infinite: the steps of their spikes are those of the network stepped one by one."""
    steps, n = 100, 130
    rng = np.random.default_rng(5)
    start = np.float32(first_step) * np.float32(dt)
    grid = (np.arange(first_step, first_step + steps + 10).astype(np.float32) * np.float32(dt)).astype(np.float32)
    trains = []
    for i in range(n):
        count = [0, 1, 3, 4, 5, 8, 9, 40, steps + 5][i % 9]
        kind = (i // 9) % 4
        if kind == 0:
            times = rng.choice(grid, count)
        elif kind == 1:
            times = np.nextafter(rng.choice(grid, count), np.float32(rng.choice([-np.inf, np.inf])))
        elif kind == 2:
            times = start + np.float32(dt) * (rng.integers(-3, steps // 10, count) * 10 + 0.5)
        else:
            times = start + np.float32(dt) * rng.uniform(-5.0, steps, count)
        times = np.sort(times.astype(np.float32))
        if count and i % 5 == 0:
            times[count // 2] = np.nan
        if count and i % 5 == 1:
            times[-1] = np.inf
        trains.append(times)
    end = np.cumsum([len(t) for t in trains])
    got = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        net = _net("dense", (n, 33), steps)
        source = net.pop("In")
        source.spike_times = np.concatenate(trains).astype(np.float32)
        source.vars = {"startSpike": np.concatenate([[0], end[:-1]]).astype(np.uint32), "endSpike": end.astype(np.uint32)}
        net.dt = dt
        model = model_from_net(net)
        model.load(num_recording_timesteps=steps)
        assert model.runner_info()["feed_forward_ahead"] == (ahead == "1")
        model.timestep = first_step
        model.run(steps)
        model.pull_recording_buffers_from_device()
        pops = [model.neuron_populations[name] for name in ("In", "Out")]
        got.append([p.vars["recordSpk"].view.copy() for p in pops] + [pops[0].vars["startSpike"].pull_from_device().copy(), pops[1].vars["V"].pull_from_device().copy()])
        model.unload()
    assert np.any(got[0][0])
    for a, b in zip(*got):
        assert np.array_equal(a, b)


# a word, one work-group's words and a few beyond, more spikes than its threads take in a round
@pytest.mark.parametrize("n", [1, 40, 32767, 32801, 70001])
def test_a_queue_cut_short_between_runs(n, monkeypatch):
    """A count written between two runs: the source's bitmap is made from the queue's first entries."""
    got = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        net = _net("dense", (n, 3), 40)
        source = net.pop("In")
        # every third neuron does not fire in the run's last step
        offset = np.where(np.arange(n) % 3 == 1, 0.0, 9.0).astype(np.float32)
        source.spike_times = np.stack([np.full(n, 4.0, np.float32), np.maximum(offset, 5.0)], axis=1).reshape(-1).astype(np.float32)
        source.vars = {"startSpike": np.arange(0, 2 * n, 2, dtype=np.uint32), "endSpike": np.arange(2, 2 * n + 2, 2, dtype=np.uint32)}
        model = model_from_net(net)
        model.load(num_recording_timesteps=40)
        assert model.runner_info()["feed_forward_ahead"] == (ahead == "1")
        model.run(10)
        source = model.neuron_populations["In"]
        left = len(source.current_spikes[0])
        assert left == np.count_nonzero(offset)
        source.vars["spkCnt"].view[:] = max(left - 3, left // 2)
        source.vars["spkCnt"].push_to_device()
        events = model.synaptic_event_count
        model.run(10)
        got.append((model.neuron_populations["Out"].vars["V"].pull_from_device().copy(), model.synaptic_event_count - events))
        model.unload()
    assert got[0][1] == got[1][1] == 3 * max(left - 3, left // 2)
    assert np.array_equal(got[0][0], got[1][0])


@pytest.mark.parametrize("kind,shape", [("dense", (65, 33)), ("conv", (5, 7, 3, 4, 3))], ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_a_recording_buffer_of_almost_2_to_the_32_rows(kind, shape):
    """The rows of a run that starts at step 0 are the first ones, however many there are said to be: steps and rows are not added up in 32 bits."""
    steps = 40
    net = _net(kind, shape, steps)
    model = model_from_net(net)
    model.load(num_recording_timesteps=steps)
    assert model.runner_info()["feed_forward_ahead"]
    oracle = OracleNet(net, num_recording_timesteps=steps)
    _abi.check(_abi.load().gennmi_run_steps(model._runner, 0, steps, 0xFFFFFFFF))
    oracle.run(steps)
    _same_rasters(net, model, oracle, steps)
    model.unload()


# fewer entries than a quad, quads that the queue's end cuts, a round of all threads' quads and one more entry, several rounds; one word, several work-groups'
# words; a second batch's queue off 16 bytes
@pytest.mark.parametrize("n, counts", [(3, (0, 1, 2, 3)), (7, (3, 4, 5, 7)), (33001, (1, 4098, 16384, 16385, 33001)), (70001, (65537, 70001))])
def test_a_queue_written_in_any_order(n, counts, monkeypatch):
    got = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        net = _net("dense", (n, 3), 40)
        source = net.pop("In")
        source.spike_times = np.zeros(1, np.float32)
        source.vars = {"startSpike": np.zeros(n, np.uint32), "endSpike": np.zeros(n, np.uint32)}
        model = model_from_net(net, batch_size=2)
        model.load(num_recording_timesteps=40)
        assert model.runner_info()["feed_forward_ahead"] == (ahead == "1")
        source = model.neuron_populations["In"]
        rng, states = np.random.default_rng(n), []
        for count in counts:
            source.vars["spk"].view.reshape(2, n)[:] = [rng.permutation(n), rng.permutation(n)]
            source.vars["spkCnt"].view[:] = [count, n - count]
            source.vars["spk"].push_to_device()
            source.vars["spkCnt"].push_to_device()
            events = model.synaptic_event_count
            model.run(8)
            states.append(model.neuron_populations["Out"].vars["V"].pull_from_device().copy())
            assert model.synaptic_event_count - events == 3 * n
        got.append(states)
        model.unload()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


# one, two and four words of rows a work-group; chunks of 64 sources without a spike at the beginning, between others, at the end and throughout
@pytest.mark.parametrize("steps", [20, 40, 100])
@pytest.mark.parametrize("active", [(), (0,), (1999,), (700, 701, 1290), tuple(range(512, 600)) + (1500,), tuple(range(0, 2000, 63))])
def test_dense_layers_of_sources_most_of_which_are_silent(steps, active, monkeypatch):
    """Every spike of the few sources counts once; among their weights are zeros, infinite ones and ones that are not a number, which keep the others
    of their groups as they are.  Sums of multiples of 2^-8 are exact: the state is that of the network stepped one by one."""
    n = 2000
    net = _net("dense", (n, 70), steps)
    source, g = net.pop("In"), net.syns[0].g.reshape(n, 70)
    trains = [np.arange(i % 3, steps - 1, 1 + i % 5, dtype=np.float32) if i in active else np.zeros(0, np.float32) for i in range(n)]
    end = np.cumsum([len(t) for t in trains])
    source.spike_times = np.concatenate(trains + [np.zeros(1, np.float32)])
    source.vars = {"startSpike": np.concatenate([[0], end[:-1]]).astype(np.uint32), "endSpike": end.astype(np.uint32)}
    for k, i in enumerate(active):
        g[i, k % 70] = [0.0, -0.0, np.inf, np.nan][k % 4]
    got = []
    for ahead in ("1", "0"):
        monkeypatch.setenv("GENNMI_AHEAD", ahead)
        model = model_from_net(net)
        model.load(num_recording_timesteps=steps)
        assert model.runner_info()["feed_forward_ahead"] == (ahead == "1")
        model.run(steps)
        model.pull_recording_buffers_from_device()
        out = model.neuron_populations["Out"]
        got.append((out.vars["V"].pull_from_device().copy(), out.vars["recordSpk"].view.copy(), model.synaptic_event_count))
        model.unload()
    assert np.array_equal(got[0][0], got[1][0], equal_nan=True) and np.array_equal(got[0][1], got[1][1])
    assert got[0][2] == got[1][2] == 70 * end[-1]


# 32 and 64 inputs a pixel and numbers off a round of 32, up to what LDS holds; few enough spikes for a list of each step, too many, and about as many as the
# rule allows; channels of one product and of two
@pytest.mark.parametrize("h,w,ic,oc,k,rate", [(9, 11, 16, 32, 3, 0.025), (9, 11, 16, 32, 3, 0.045), (12, 6, 8, 7, 3, 0.04), (10, 9, 7, 34, 3, 0.06), (8, 9, 16, 3, 2, 0.05),
                                              (7, 7, 13, 5, 5, 0.012), (7, 8, 19, 4, 5, 0.01), (9, 9, 8, 32, 2, 0.05), (11, 33, 4, 33, 5, 0.03)])
@pytest.mark.parametrize("steps", [8, 32, 45])
def test_sums_of_convolutions_with_few_spikes(h, w, ic, oc, k, rate, steps):
    """A step's sum is that of its inputs' weights in the kernel's order, whichever way it is made: outPost bit for bit as 32-bit sums in that order give it.
    Two pixels have steps with 15, 16 and 17 inputs (a list holds 16), and one step has no spike at all."""
    rng = np.random.default_rng(h * w + steps)
    net = configs.conv_toeplitz(h=h, w=w, ic=ic, oc=oc, k=k, steps=steps, w_sd=0.1, ioffset=0.3)
    fire = rng.random((steps, h, w, ic)) < rate
    before, after = (k - 1) - (k - 1) // 2, (k - 1) // 2
    for step, y, x, count in ((1, 4, 4, 15), (3, 4, 4, 16), (5, 4, 4, 17), (5, 5, 3, 16), (6, 2, 4, 17)):
        patch = np.zeros((min(k, 4), min(k, 4), ic), bool).reshape(-1)
        patch[rng.permutation(len(patch))[:count]] = True
        side = min(k, 4)
        fire[step, y - before:y - before + side, x - before:x - before + side] = patch.reshape(side, side, ic)
    fire[2] = False
    trains = fire.reshape(steps, -1).T
    end = np.cumsum(trains.sum(axis=1)).astype(np.uint32)
    source = net.pop("In")
    source.vars = {"startSpike": (end - trains.sum(axis=1)).astype(np.uint32), "endSpike": end}
    source.spike_times = np.nonzero(trains)[1].astype(np.float32)
    model = model_from_net(net)
    model.load(num_recording_timesteps=steps)
    assert model.runner_info()["feed_forward_ahead"]
    model.run(steps)
    got = model.synapse_populations["Conv"].vars["outPost"].pull_from_device().copy()
    model.unload()
    want = np.zeros((h, w, oc), np.float32)
    decay = np.float32(np.exp(-1.0 / 5.0))
    kernel = net.syns[0].g
    for step in range(steps):
        sums = np.zeros((h, w, oc), np.float32)
        if step:
            padded = np.pad(fire[step - 1], ((before, after), (before, after), (0, 0)))
            for a in range(k):
                for b in range(k):
                    for channel in range(ic):
                        sums += np.where(padded[a:a + h, b:b + w, channel, None], kernel[a, b, channel], np.float32(0))
        want = (want + sums) * decay
    assert np.array_equal(got.reshape(want.shape).view(np.uint32), want.view(np.uint32))


# fewer than 32 inputs a pixel (lists of four), and two output rows a work-group
@pytest.mark.parametrize("h,w,ic,oc,k,rate", [(9, 11, 1, 5, 5, 0.06), (9, 11, 2, 32, 3, 0.08), (64, 6, 4, 1056, 3, 0.03)])
@pytest.mark.parametrize("steps", [8, 32, 45])
def test_sums_of_convolutions_with_short_lists(h, w, ic, oc, k, rate, steps):
    """The same where a list holds fewer than 16 inputs."""
    test_sums_of_convolutions_with_few_spikes(h, w, ic, oc, k, rate, steps)
