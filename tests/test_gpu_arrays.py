"""What a program may hand to arrays and look at on their host side."""
import numpy as np
import pytest

from genn_amd import _abi, configs, genn_model
from genn_amd.genn_model import init_postsynaptic, init_weight_update, model_from_net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("fires", ["pre", "post"])
def test_initial_traces_may_be_one_a_neuron(make_model, fires, batch):
    """A spike of one side meets the other side's traces: weights move by exactly these (no decay, traces are eighths)."""
    n_pre, n_post, rng = 70, 130, np.random.default_rng(3)
    traces = {"pre": rng.integers(1, 64, batch * n_pre).astype(np.float64) / 8.0, "post": rng.integers(1, 64, batch * n_post) / 8.0}
    m = make_model("float", "traces", dt=1.0, batch_size=batch)
    pops = {}
    for name, n in (("pre", n_pre), ("post", n_post)):
        end = np.arange(1, n + 1) if name == fires else np.zeros(n)
        pops[name] = m.add_neuron_population(name, n, "SpikeSourceArray", {}, {"startSpike": np.maximum(end - 1, 0), "endSpike": end})
        pops[name].set_extra_global_param("spikeTimes", np.zeros(n, np.float32))
    stdp = {"tauPlus": 1e30, "tauMinus": 1e30, "aPlus": 1.0, "aMinus": 1.0, "wMin": -100.0, "wMax": 100.0}
    s = m.add_synapse_population("S", "SPARSE", pops["pre"], pops["post"],
                                 init_weight_update("STDPTrace", stdp, {"g": 0.0}, {"preTrace": traces["pre"]}, {"postTrace": traces["post"]}),
                                 init_postsynaptic("DeltaCurr"))
    i, j = np.nonzero(rng.random((n_pre, n_post)) < 0.3)
    s.set_sparse_connections(i, j)
    m.build()
    m.load()
    for var, name in (("preTrace", "pre"), ("postTrace", "post")):
        assert np.array_equal(s.vars[var].view, traces[name].astype(np.float32))
        assert np.array_equal(s.vars[var].pull_from_device(), traces[name].astype(np.float32))
    m.step_time()
    m.step_time()
    moved = s.vars["g"].pull_from_device().reshape(batch, n_pre, s.row_stride)
    for b in range(batch):
        want = traces["pre"].reshape(batch, n_pre)[b][i] if fires == "post" else -traces["post"].reshape(batch, n_post)[b][j]
        assert np.array_equal(moved[b][np.arange(s.row_stride)[None, :] < s.row_length_host[:, None]], want.astype(np.float32))


@pytest.mark.parametrize("fill", [2.5, np.float32(2.5), np.array(2.5), [2.5], np.arange(5.0), [1, 2, 3, 4, 5]])
def test_an_arrays_first_value_is_one_of_all_or_one_each(fill):
    _abi.check(_abi.load().gennmi_init(0))
    a = genn_model.Array(5, np.float32, fill=fill)
    want = np.full(5, fill, dtype=np.float32)
    assert np.array_equal(a.pull_slice(0, 5), want)
    assert np.array_equal(a.view, want) and np.array_equal(a.pull_from_device(), want)
    a.free()


@pytest.mark.parametrize("batch, delay", [(1, 0), (3, 0), (1, 3), (2, 2)])
def test_current_spikes_leaves_the_queue_on_the_host_side(make_model, batch, delay):
    """After current_spikes the host sides of `spkCnt` and `spk` show what the device's hold, in arrays a program may have kept."""
    n, steps, rng = 300, 8, np.random.default_rng(11)
    fire = rng.random((batch, n, steps)) < 0.2
    fire[:, :, 3] = False
    fire[:, :, 5] = True
    count = fire.sum(axis=2).reshape(-1)
    end = np.cumsum(count).reshape(batch, n)
    m = make_model("float", "queues", dt=1.0, batch_size=batch)
    src = m.add_neuron_population("S", n, "SpikeSourceArray", {}, {"startSpike": end - count.reshape(batch, n), "endSpike": end})
    src.set_extra_global_param("spikeTimes", np.nonzero(fire.reshape(batch * n, steps))[1].astype(np.float32))
    lif = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=1e9, Ioffset=0.0, TauRefrac=5.0)
    trg = m.add_neuron_population("T", 5, "LIF", lif, {"V": -60.0, "RefracTime": 0.0})
    s = m.add_synapse_population("ST", "SPARSE", src, trg, init_weight_update("StaticPulse", {}, {"g": 1.0}), init_postsynaptic("DeltaCurr"))
    s.set_sparse_connections([0, 1], [0, 1])
    s.axonal_delay_steps = delay
    m.build()
    m.load()
    slots = src.num_delay_slots
    assert slots == (delay + 1 if delay else 1)
    kept = src.vars["spkCnt"].view, src.vars["spk"].view
    for step in range(steps):
        m.step_time()
        spikes = src.current_spikes
        counts, ids = src.vars["spkCnt"].view, src.vars["spk"].view
        assert counts is kept[0] and ids is kept[1]
        assert np.array_equal(counts, src.vars["spkCnt"].pull_slice(0, batch * slots))
        device = src.vars["spk"].pull_slice(0, batch * slots * n).reshape(-1, n)
        for q, c in enumerate(counts):
            assert np.array_equal(ids.reshape(-1, n)[q, :c], device[q, :c])
        for b in range(batch):
            assert np.array_equal(spikes[b], np.nonzero(fire[b, :, step])[0])
            assert not np.shares_memory(spikes[b], ids)


def _run_of_a_small_network():
    """Everything that is copied: pushes and pulls of small and large arrays, queues of one slot and of several, recordings, a copy on the device."""
    m = model_from_net(configs.vogels_abbott(n=2000, steps=40, p=0.05, axonal_delays={"EI": 3}), ordered=True)     # (sums in a fixed order)
    batched = model_from_net(configs.conv_toeplitz(h=16, w=16, ic=4, oc=8, steps=10, max_rate=300.0), batch_size=2)
    out = []
    for model, steps in ((m, 40), (batched, 10)):
        model.load(num_recording_timesteps=steps)
        for _ in range(steps):
            model.step_time()
            out += [ids for p in model.neuron_populations.values() for ids in p.current_spikes]
        model.pull_recording_buffers_from_device()
        out += [p.vars["recordSpk"].view.copy() for p in model.neuron_populations.values()]
    a, b = m._alloc(1_300_001, np.float32), m._alloc(1_300_001, np.float32)
    a.view[:] = np.arange(a.count)
    a.push_to_device()
    b.copy_on_device(a)
    out += [b.pull_from_device().copy()] + [p.vars["V"].pull_from_device().copy() for p in m.neuron_populations.values()]
    for model in (m, batched):
        model.unload()
    return out


def test_copies_without_pinned_memory(monkeypatch):
    """Where none is to be had the host sides are ordinary memory and the runtime's copies move everything: the same bytes."""
    _abi.check(_abi.load().gennmi_init(0))
    want = _run_of_a_small_network()
    monkeypatch.setenv("GENNMI_PINNED_COPIES", "0")
    _abi.check(_abi.load().gennmi_release_cached_memory())      # (also the staging memory of earlier copies)
    a = genn_model.Array(10, np.float32, pinned=True)
    assert a.view.base is None          # (its own memory, nothing of the library's)
    a.free()
    got = _run_of_a_small_network()
    monkeypatch.delenv("GENNMI_PINNED_COPIES")
    assert len(want) == len(got) and sum(int(np.any(w)) for w in want) > 20
    assert all(np.array_equal(w, g) for w, g in zip(want, got))
    again = _run_of_a_small_network()
    assert all(np.array_equal(w, g) for w, g in zip(want, again))


def test_a_refused_host_side_is_ordinary_memory(make_model, monkeypatch):
    lib = _abi.load()
    _abi.check(lib.gennmi_init(0))
    monkeypatch.setattr(genn_model, "_Pinned", lambda count, dtype: _abi.check(2))
    a = genn_model.Array(1000, np.float32, fill=3.0, pinned=True)
    assert np.array_equal(a.pull_from_device(), np.full(1000, 3.0, np.float32))
    a.view[:] = 4.0
    a.push_to_device()
    assert np.array_equal(a.pull_slice(0, 1000), a.view)
    a.free()


@pytest.mark.parametrize("looked_at_before", [False, True])
def test_given_values_are_there_after_unload(looked_at_before):
    m = genn_model.GeNNModel("float", "noise", dt=1.0)
    pop = m.add_neuron_population("N", 40, "LIF", dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=0.0, TauRefrac=5.0), {"V": -60.0, "RefracTime": 0.0})
    noise = np.random.default_rng(5).random((3, 40)).astype(np.float32)
    source = m.add_current_source("noise", "ArrayNoise", pop)
    source.set_extra_global_param("noise", noise)
    m.build()
    m.load()
    if looked_at_before:
        assert np.array_equal(source.vars["noise"].view, noise.reshape(-1))
    m.unload()
    assert np.array_equal(source.vars["noise"].view, noise.reshape(-1))
