"""Device memory kept between models, and the segment boundaries built with the tables of a new one."""
import ctypes as C
import threading
import time

import numpy as np
import pytest
import torch

from genn_amd import _abi, configs
from genn_amd.genn_model import (Array, GeNNModel, init_postsynaptic, init_sparse_connectivity, init_var, init_weight_update, model_from_net,
                                 release_cached_memory)

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _malloc(lib, nbytes):
    p = C.c_void_p()
    _abi.check(lib.gennmi_malloc(C.byref(p), nbytes))
    return p


def test_blocks_are_kept_by_size_and_given_back():
    lib = _abi.load()
    _abi.check(lib.gennmi_init(0))
    _abi.check(lib.gennmi_release_cached_memory())
    a, b = _malloc(lib, 40 * MIB), _malloc(lib, 41 * MIB)
    assert a.value != b.value
    for p in (a, b):
        _abi.check(lib.gennmi_free(p))
    c = _malloc(lib, 41 * MIB)          # (the smallest kept block it fits)
    d = _malloc(lib, 38 * MIB)          # (within an eighth of the block's size)
    e = _malloc(lib, 38 * MIB)          # (none left)
    assert (c.value, d.value) == (b.value, a.value) and e.value not in (a.value, b.value)
    for p in (c, d, e):
        _abi.check(lib.gennmi_free(p))
    kept, left = C.c_size_t(), C.c_size_t()
    _abi.check(lib.gennmi_free_device_memory_bytes(C.byref(kept)))
    _abi.check(lib.gennmi_release_cached_memory())
    _abi.check(lib.gennmi_free_device_memory_bytes(C.byref(left)))
    assert abs(kept.value - left.value) <= 64 * MIB


def test_kept_blocks_under_threads():
    """Every thread sees its own bytes: a block in use is never handed out twice."""
    lib = _abi.load()
    _abi.check(lib.gennmi_init(0))
    failures = []

    def work(k):
        rng = np.random.default_rng(k)
        for _ in range(8):
            count = int(rng.integers(600_000, 700_000))
            a = Array(count, np.float32, fill=float(k))
            got = a.pull_slice(count - 1000, 1000)
            if not np.all(got == k):
                failures.append((k, got))
            a.free()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


def _pooled(m):
    return {v.ptr for g in (m.neuron_populations, m.synapse_populations) for p in g.values() for v in p.vars.values() if v.count * v.dtype.itemsize >= 2 * MIB}


def _plastic(seed):
    return model_from_net(configs.plastic_stdp(n=5000, n_src=50, steps=60, fan=400, src_fan=100, seed=seed)), 60


def _device_made(seed):
    """Matrices made on the device, rows of different lengths (what lies behind a row's end is nobody's); sums of halves, exact in any order."""
    m = GeNNModel("float", "made", dt=1.0)
    m.seed = seed
    lif = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=0.55, TauRefrac=5.0)
    pops = {k: m.add_neuron_population(k, n, "LIF", lif, {"V": init_var("Uniform", {"min": -60.0, "max": -50.0}), "RefracTime": 0.0})
            for k, n in (("E", 20000), ("I", 5003))}
    for src, w in (("E", 0.5), ("I", -2.0)):
        for trg in "EI":
            m.add_synapse_population(src + trg, "SPARSE", pops[src], pops[trg], init_weight_update("StaticPulse", {}, {"g": init_var("Constant", {"constant": w})}),
                                     init_postsynaptic("DeltaCurr"), init_sparse_connectivity("FixedProbability", {"prob": 0.015}))
    for p in pops.values():
        p.spike_recording_enabled = True
    m.build()
    return m, 60


@pytest.mark.parametrize("model", [_plastic, _device_made])
def test_models_one_after_another_are_the_same(model):
    """A model built from kept blocks that are full of another one's values (its indices are in range here) runs as the first one did."""
    release_cached_memory()
    runs, blocks = [], []
    for seed in (99, 100, 99, 101, 99):
        m, steps = model(seed)
        m.load(num_recording_timesteps=steps)
        m.run(steps)
        m.pull_recording_buffers_from_device()
        runs.append([p.vars["recordSpk"].view.copy() for p in m.neuron_populations.values()])
        blocks.append(_pooled(m))
        m.unload()
    first, others = runs[0], (runs[1], runs[3])
    assert sum(int(a.sum() != 0) for a in first) > 0
    for r in (runs[2], runs[4]):
        assert all(np.array_equal(a, b) for a, b in zip(first, r))
    for r in others:            # (another model indeed, in the same blocks)
        assert any(not np.array_equal(a, b) for a, b in zip(first, r))
    assert blocks[0] and all(b & blocks[0] for b in blocks[1:])


@pytest.mark.parametrize("n_trg, tile_floats", [(1, 16), (63, 16), (64, 16), (100, 7), (4097, 1024), (3000, 1000)])
@pytest.mark.parametrize("row_len", [0, 1, 63, 64, 65, 130])
def test_tile_path_sums_at_row_and_tile_edges(n_trg, tile_floats, row_len, monkeypatch):
    """Rows around a wavefront's 64 synapses, targets around tile boundaries (power of two and not): integer weights, exact sums."""
    monkeypatch.setenv("GENNMI_TILE_FLOATS", str(tile_floats))
    n_src, rng = 70, np.random.default_rng(n_trg * 131 + row_len)
    rows = [np.sort(rng.integers(0, n_trg, row_len if r else n_trg if n_trg < 200 else 200)) for r in range(n_src)]
    pre = np.concatenate([np.full(len(r), k) for k, r in enumerate(rows)])
    post = np.concatenate(rows)
    m = GeNNModel("float", "edges", dt=1.0)
    src = m.add_neuron_population("S", n_src, "SpikeSourceArray", {}, {"startSpike": np.arange(n_src), "endSpike": np.arange(n_src) + 1})
    src.set_extra_global_param("spikeTimes", np.zeros(n_src, np.float32))
    trg = m.add_neuron_population("T", n_trg, "LIF", dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=1e9, Ioffset=0.0, TauRefrac=5.0),
                                  {"V": -60.0, "RefracTime": 0.0})
    s = m.add_synapse_population("ST", "SPARSE", src, trg, init_weight_update("StaticPulse", {}, {"g": 0.0}), init_postsynaptic("DeltaCurr"))
    s.set_sparse_connections(pre, post)
    weights = rng.integers(-8, 9, len(pre)).astype(np.float32)
    s.set_var_coo("g", weights)
    m.build()
    m.load()
    m.step_time()               # every source fires in the first step
    m.update_synapses()
    want = np.zeros(n_trg, np.float32)
    np.add.at(want, post, weights)
    assert np.array_equal(s.vars["outPost"].pull_from_device(), want)
    m.unload()


def _gib_in_use():
    """Device memory in use, in whole GiB over or under a start: the runtime's own few MiB come and go between two looks."""
    free, total = torch.cuda.mem_get_info()
    return (total - free) / 1024.0 ** 3


def test_kept_memory_goes_back_by_itself(monkeypatch):
    """A process that frees and then does nothing gives kept memory back when its time has come; what is asked for before is a kept block."""
    _abi.check(_abi.load().gennmi_init(0))
    release_cached_memory()
    before, size = _gib_in_use(), 1024 * MIB
    monkeypatch.setenv("GENNMI_POOL_SECONDS", "0.5")
    lib = _abi.load()
    kept = _malloc(lib, size)
    _abi.check(lib.gennmi_free(kept))
    assert round(_gib_in_use() - before) == 1
    again = _malloc(lib, size)
    assert again.value == kept.value
    time.sleep(0.7)             # (in use: its time does not run)
    assert round(_gib_in_use() - before) == 1
    _abi.check(lib.gennmi_free(again))
    deadline = time.monotonic() + 20.0
    while round(_gib_in_use() - before) and time.monotonic() < deadline:
        time.sleep(0.05)
    assert round(_gib_in_use() - before) == 0
    monkeypatch.setenv("GENNMI_POOL_SECONDS", "0")
    _abi.check(lib.gennmi_free(_malloc(lib, size)))
    assert round(_gib_in_use() - before) == 0


def test_release_cached_memory_gives_everything_back():
    _abi.check(_abi.load().gennmi_init(0))
    release_cached_memory()
    before = _gib_in_use()
    arrays = [Array(64 << 20, np.float32, fill=1.0) for _ in range(4)]
    for a in arrays:
        a.free()
    assert round(_gib_in_use() - before) == 1
    release_cached_memory()
    assert round(_gib_in_use() - before) == 0


def test_memory_goes_back_while_models_step_and_threads_allocate(monkeypatch):
    """The thread that gives blocks back runs beside steps, copies and allocations: nobody's values change."""
    monkeypatch.setenv("GENNMI_POOL_SECONDS", "0.01")
    m, steps = _device_made(99)
    m.load(num_recording_timesteps=steps)
    m.run(steps)
    m.pull_recording_buffers_from_device()
    want = [p.vars["recordSpk"].view.copy() for p in m.neuron_populations.values()]
    m.unload()
    failures, stop = [], threading.Event()

    def work(k):
        rng = np.random.default_rng(k)
        while not stop.is_set():
            count = int(rng.integers(600_000, 2_000_000))
            a = Array(count, np.float32, fill=float(k), pinned=True)
            a.pull_from_device()
            if not (a.view[0] == a.view[-1] == k):
                failures.append(k)
            a.free()
            time.sleep(float(rng.uniform(0.0, 0.02)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    try:
        for _ in range(8):
            m, _ = _device_made(99)
            m.load(num_recording_timesteps=steps)
            for _ in range(steps):
                m.step_time()
            m.pull_recording_buffers_from_device()
            assert all(np.array_equal(p.vars["recordSpk"].view, w) for p, w in zip(m.neuron_populations.values(), want))
            m.unload()
    finally:
        stop.set()
        for t in threads:
            t.join()
    assert not failures


def test_memory_goes_back_beside_a_capture(monkeypatch):
    """Giving a block back waits for the device, which a stream that somebody is capturing must not notice."""
    _abi.check(_abi.load().gennmi_init(0))
    release_cached_memory()
    lib, size = _abi.load(), 1024 * MIB
    x = torch.arange(1000, dtype=torch.float32, device="cuda")
    y = x * 2.0                 # (compiled and allocated before the capture)
    torch.cuda.synchronize()
    before = _gib_in_use()
    monkeypatch.setenv("GENNMI_POOL_SECONDS", "0.3")
    kept = _malloc(lib, size)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _abi.check(lib.gennmi_free(kept))       # (kept, not freed: nothing of the runtime's is called)
        time.sleep(0.8)
        y = x * 3.0
    deadline = time.monotonic() + 20.0
    while round(_gib_in_use() - before) and time.monotonic() < deadline:
        time.sleep(0.05)
    assert round(_gib_in_use() - before) == 0
    for k in range(3):
        x.fill_(float(k))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.all(y == 3.0 * k)
