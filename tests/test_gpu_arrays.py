"""What a program may hand to arrays and look at on their host side."""
import numpy as np
import pytest

from genn_amd.genn_model import init_postsynaptic, init_weight_update

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
    from genn_amd import _abi
    from genn_amd.genn_model import Array
    _abi.check(_abi.load().gennmi_init(0))
    a = Array(5, np.float32, fill=fill)
    want = np.full(5, fill, dtype=np.float32)
    assert np.array_equal(a.pull_slice(0, 5), want)
    assert np.array_equal(a.view, want) and np.array_equal(a.pull_from_device(), want)
    a.free()
