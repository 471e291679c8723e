"""The resident plan (many timesteps per launch; neuron state in registers, delay rings in LDS, tiles exchanging their
spikes through one word each) against the CPU oracle, on the paths the benchmark networks do not reach often:
segments with more due synapses than an entry holds inline, steps with more (spike, projection) pairs than a tile
stages at once, tiles with many spikes in one step (side buffer), weights pushed between launches.

Weights are one value per projection and every postsynaptic model has one incoming projection, so no fp32 sum depends
on the order of its additions and everything — state, rings, spike queues, recordings, event counts — must be identical.
"""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

from genn_amd import _abi, rng
from genn_amd.genn_model import model_from_net, release_cached_memory
from genn_amd.netspec import CurrentSource, Net, Pop, Syn
from oracle.genn_cpu import OracleNet
from parity import compare_state

pytestmark = pytest.mark.gpu

LIF = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=0.0, TauRefrac=2.0)


def _pop(name, n, ioffset, v0):
    return Pop(name, "lif", n, dict(LIF, Ioffset=ioffset), {"V": np.asarray(v0, np.float32), "RefracTime": np.zeros(n, np.float32)})


def _projection(name, src, trg, n_src, n_trg, stride, weight, seed, depth=0, due_share=0.0, tau=5.0):
    """Random ascending rows of exactly `stride` targets; with depth > 0 a dendritic delay per synapse, a share
    `due_share` of which is a multiple of the ring depth (those land in the slot read in the step that delivers them)."""
    ind = np.sort(rng.randint(seed, 1, 0, n_src * stride, n_trg).reshape(n_src, stride), axis=1).astype(np.uint32)
    syn = Syn(name, src, trg, wum="static_delay" if depth else "static", psm="expcurr", tau=tau, row_stride=stride,
              row_length=np.full(n_src, stride, np.uint32), ind=ind, g=np.full((n_src, stride), weight, np.float32))
    if depth:
        u = rng.uniform(seed, 2, 0, n_src * stride).reshape(n_src, stride)
        later = 1 + rng.randint(seed, 3, 0, n_src * stride, depth - 1).reshape(n_src, stride)
        syn.d = np.where(u < due_share, 0, later).astype(np.uint8)
        syn.max_den_delay = depth
    return syn


def _run_chunks(net, chunks, check, resident=True):
    model = model_from_net(net)
    steps = sum(chunks)
    model.load(num_recording_timesteps=steps)
    assert model.runner_info()["resident_plan"] == resident
    oracle = OracleNet(net, num_recording_timesteps=steps)
    for chunk in chunks:
        if chunk < 0:                       # eager single steps in between
            for _ in range(-chunk):
                model.step_time()
            oracle.run(-chunk)
        else:
            model.run(chunk)
            oracle.run(chunk)
        model.synchronize()
        check(model, oracle)
    model.pull_recording_buffers_from_device()
    spikes = 0
    for p in net.pops:
        want = oracle.record(p.name, steps)
        assert np.array_equal(model.neuron_populations[p.name].vars["recordSpk"].view, want), f"recording of {p.name} differs"
        assert np.array_equal(model.neuron_populations[p.name].current_spikes[0], oracle.spikes(p.name))
        spikes += int(np.unpackbits(want.view(np.uint8)).sum())
    assert model.synaptic_event_count == oracle.events()
    return model, oracle, spikes


@pytest.mark.parametrize("due_share", [0.5, 0.04, 1.0])
def test_due_synapses_inline_and_row_walk(due_share):
    """Delayed projections between two populations of 700 and 300 neurons (3 + 2 tiles, ragged last tiles).  With half of
    the delays a multiple of the ring depth nearly every segment has more due synapses than fit inline (row walk before
    the update); with 4 % most have none or a few (inline); with all of them due nothing is left for later."""
    n_a, n_b, depth = 700, 300, 7
    net = Net(name="resident_due", dt=1.0, steps=0)
    net.pops.append(_pop("A", n_a, 0.62, -60.0 + 9.5 * rng.uniform(5, 1, 0, n_a)))
    net.pops.append(_pop("B", n_b, 0.45, -60.0 + 9.5 * rng.uniform(5, 2, 0, n_b)))
    net.syns.append(_projection("AB", "A", "B", n_a, n_b, 40, 0.11, 11, depth, due_share))
    net.syns.append(_projection("BA", "B", "A", n_b, n_a, 64, -0.07, 12, depth, due_share))
    net.syns.append(_projection("AA", "A", "A", n_a, n_a, 24, 0.05, 13, depth, due_share, tau=9.0))
    net.steps = 260

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)

    # launches of 100, 5 and 60 steps with eager single steps (the one-launch-per-step plan) in between
    model, oracle, spikes = _run_chunks(net, (100, -3, 5, -2, 60, 90), check)
    assert model.runner_info()["single_launch_step"]
    assert spikes > 2000
    model.unload()


@pytest.mark.parametrize("depth", [0, 5])
def test_more_pairs_than_a_tile_stages(depth):
    """3,000 neurons cross threshold in the same step: every tile of the target sees 3,000 (spike, projection) pairs in one
    exchange, more than it stages at once, and every source tile sends 256 spikes through the side buffer."""
    n_a, n_b = 3000, 520
    net = Net(name="resident_burst", dt=1.0, steps=0)
    net.pops.append(_pop("A", n_a, 1.0, np.full(n_a, -50.4)))
    net.pops.append(_pop("B", n_b, 0.3, np.full(n_b, -58.0)))
    net.syns.append(_projection("AB", "A", "B", n_a, n_b, 12, 0.002, 21, depth, 0.3))
    net.syns.append(_projection("BA", "B", "A", n_b, n_a, 30, -0.05, 22, depth, 0.3))
    net.steps = 80

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)

    model, oracle, spikes = _run_chunks(net, (6, 34, 40), check)
    first = oracle.record("A", 80).reshape(80, -1)[0]
    assert int(np.unpackbits(first.view(np.uint8)).sum()) == n_a          # the burst happened in step 0
    assert spikes > 2 * n_a
    model.unload()


@pytest.mark.parametrize("n_a, ioffset, targets", [(400, 1.0, 120), (24, 0.62, 120), (12, 0.62, 120), (400, 1.0, 14), (24, 0.62, 64), (12, 0.62, 50), (12, 0.62, 65)])
def test_long_row_parts_take_several_trips(n_a, ioffset, targets):
    """Rows inside one tile of 200 neurons.  A lane reads four synapses of its pair's part in one trip to memory: a pair has 4 lanes and 16 synapses
    a trip when many pairs are listed (400 sources crossing threshold together), 16 lanes and 64 synapses when few are (24 or 12 sources firing
    now and then).  Parts of 120 and 65 take several trips, parts of 14, 50 and 64 take one."""
    n_b, depth = 200, 6
    net = Net(name="resident_long_parts", dt=1.0, steps=0)
    v0 = np.full(n_a, -50.4) if n_a == 400 else -60.0 + 9.5 * rng.uniform(41, 1, 0, n_a)
    net.pops.append(_pop("A", n_a, ioffset, v0))
    net.pops.append(_pop("B", n_b, 0.3, np.full(n_b, -58.0)))
    net.syns.append(_projection("AB", "A", "B", n_a, n_b, targets, 0.004 if n_a == 400 else 0.05, 42, depth, 0.1))
    net.steps = 90

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)

    model, oracle, spikes = _run_chunks(net, (30, 60), check)
    assert spikes > (n_a if n_a == 400 else 20)
    model.unload()


def test_pushed_weights_reach_the_inline_copies(monkeypatch):
    """The segment tables hold copies of the weights of due synapses; a push of `g` between launches must refresh them.
    (With the one-launch-per-step plan the due synapses of the last step's spikes are already in the ring when the push
    happens — at their old weights, where the reference would add them after the push — so that plan is switched off
    here: the test is about the copies.)"""
    monkeypatch.setenv("GENNMI_FUSED_STEP", "0")
    n, depth = 600, 4
    net = Net(name="resident_push", dt=1.0, steps=0)
    net.pops.append(_pop("A", n, 0.6, -60.0 + 9.5 * rng.uniform(7, 1, 0, n)))
    net.syns.append(_projection("AA", "A", "A", n, n, 48, 0.04, 31, depth, 0.4))
    net.steps = 120

    state = {"pushed": False}

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)
        if not state["pushed"]:
            g = model.synapse_populations["AA"].vars["g"]
            g.view[:] = np.float32(-0.03)
            g.push_to_device()
            oracle.syn_g("AA")[:] = np.float32(-0.03)
            state["pushed"] = True

    model, oracle, spikes = _run_chunks(net, (60, 60), check)
    assert spikes > 500
    model.unload()


def test_weights_written_behind_the_library_are_reported(monkeypatch):
    """A caller that overwrites `g` by its own means (here: a device-to-device copy the runner is not told about) and then
    names the range with gennmi_note_device_write gets the same refresh of the inline copies and packed records as a push."""
    import ctypes as C
    from genn_amd import _abi
    monkeypatch.setenv("GENNMI_FUSED_STEP", "0")
    n, depth = 600, 4
    net = Net(name="resident_note", dt=1.0, steps=0)
    net.pops.append(_pop("A", n, 0.6, -60.0 + 9.5 * rng.uniform(7, 1, 0, n)))
    net.syns.append(_projection("AA", "A", "A", n, n, 48, 0.04, 31, depth, 0.4))
    net.steps = 120
    state = {"written": False}

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)
        if not state["written"]:
            g = model.synapse_populations["AA"].vars["g"]
            lib = _abi.load()
            staging = C.c_void_p()
            _abi.check(lib.gennmi_malloc(C.byref(staging), g.view.nbytes))
            new = np.full(g.count, -0.03, np.float32)
            _abi.check(lib.gennmi_memcpy_to_device(staging, new.ctypes.data_as(C.c_void_p), new.nbytes))
            hip = C.CDLL("libamdhip64.so")
            assert hip.hipMemcpy(C.c_void_p(g.ptr), staging, C.c_size_t(new.nbytes), C.c_int(3)) == 0      # hipMemcpyDeviceToDevice
            _abi.check(lib.gennmi_note_device_write(C.c_void_p(g.ptr), new.nbytes))
            lib.gennmi_free(staging)
            oracle.syn_g("AA")[:] = np.float32(-0.03)
            state["written"] = True

    model, oracle, spikes = _run_chunks(net, (60, 60), check)
    assert spikes > 500
    model.unload()


def test_writes_named_through_a_registered_host_buffer(monkeypatch):
    """The same for callers that only know host pointers (generated custom update code beside the library's kernels): the
    device buffer is registered behind a host buffer, gennmi_flush runs queued steps before the caller's own device work, and
    gennmi_note_mirror_write names the whole device buffer through any pointer into the host one.  One of two projections is
    rewritten: only its copies are rebuilt, and the other one's stay valid."""
    import ctypes as C
    from genn_amd import _abi
    monkeypatch.setenv("GENNMI_FUSED_STEP", "0")
    n, depth = 600, 4
    net = Net(name="resident_mirror", dt=1.0, steps=0)
    net.pops.append(_pop("A", n, 0.6, -60.0 + 9.5 * rng.uniform(17, 1, 0, n)))
    net.syns.append(_projection("AA", "A", "A", n, n, 48, 0.04, 31, depth, 0.4))
    net.syns.append(_projection("AA2", "A", "A", n, n, 24, -0.02, 41, depth, 0.3))
    net.steps = 120
    state = {"written": False, "host": None}

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)
        if not state["written"]:
            g = model.synapse_populations["AA"].vars["g"]
            lib = _abi.load()
            host = np.zeros(g.count, np.float32)                       # the caller's host buffer (never copied from here)
            state["host"] = host
            _abi.check(lib.gennmi_register_mirror(host.ctypes.data_as(C.c_void_p), C.c_void_p(g.ptr), host.nbytes))
            _abi.check(lib.gennmi_flush())
            staging = C.c_void_p()
            _abi.check(lib.gennmi_malloc(C.byref(staging), host.nbytes))
            new = np.full(g.count, -0.03, np.float32)
            _abi.check(lib.gennmi_memcpy_to_device(staging, new.ctypes.data_as(C.c_void_p), new.nbytes))
            hip = C.CDLL("libamdhip64.so")
            assert hip.hipMemcpy(C.c_void_p(g.ptr), staging, C.c_size_t(new.nbytes), C.c_int(3)) == 0      # hipMemcpyDeviceToDevice
            _abi.check(lib.gennmi_note_mirror_write(C.c_void_p(host.ctypes.data + 4 * 100)))               # a pointer INTO the host buffer
            lib.gennmi_free(staging)
            assert lib.gennmi_note_mirror_write(C.c_void_p(new.ctypes.data)) != 0                           # not a registered buffer
            _abi.check(lib.gennmi_unregister_mirror(host.ctypes.data_as(C.c_void_p)))
            oracle.syn_g("AA")[:] = np.float32(-0.03)
            state["written"] = True

    model, oracle, spikes = _run_chunks(net, (60, 60), check)
    assert model.runner_info()["resident_plan"]
    assert spikes > 500
    model.unload()


@pytest.mark.parametrize("limit, rows", [(64, 230), (1000, 230), (7, 230), (64, 50), (64, 0)])
def test_queued_single_steps_take_the_resident_launch(limit, rows):
    """step_time() one call at a time with the step queue on (what the reference's Runtime::stepTime amounts to): the steps
    run as resident launches of up to `limit` steps, cut wherever something looks at the device -- state pulls, a push
    of membrane potentials, the event counter, a recording buffer of `rows` rows that wraps -- and everything is as unqueued stepping leaves it."""
    n_a, n_b, depth = 700, 300, 7
    net = Net(name="resident_queue", dt=1.0, steps=230)
    net.pops.append(_pop("A", n_a, 0.62, -60.0 + 9.5 * rng.uniform(5, 1, 0, n_a)))
    net.pops.append(_pop("B", n_b, 0.45, -60.0 + 9.5 * rng.uniform(5, 2, 0, n_b)))
    net.syns.append(_projection("AB", "A", "B", n_a, n_b, 40, 0.11, 11, depth, 0.3))
    net.syns.append(_projection("BA", "B", "A", n_b, n_a, 64, -0.07, 12, depth, 0.3))
    model = model_from_net(net, record=bool(rows))
    model.load(num_recording_timesteps=rows or None)
    assert model.runner_info()["resident_plan"]
    model.set_step_queue(limit)
    oracle = OracleNet(net, num_recording_timesteps=rows)
    done = 0
    for chunk in (1, 2, 3, 40, 9, 100, 75):
        for _ in range(chunk):
            model.step_time()
        oracle.run(chunk)
        done += chunk
        if done == 55:
            # a push lands between the steps it was issued between (the steps queued before it have run by then)
            v = model.neuron_populations["B"].vars["V"]
            v.pull_from_device()
            v.view[::3] = np.float32(-50.5)
            v.push_to_device()
            oracle.var("B", 0)[::3] = np.float32(-50.5)
        elif done == 155:
            assert model.synaptic_event_count == oracle.events()
        else:
            compare_state(net, model, oracle, f"after {done} queued steps", exact=True)      # pulls, no synchronize() first
    assert done == net.steps
    if rows:
        model.pull_recording_buffers_from_device()
        for p in net.pops:
            assert np.array_equal(model.neuron_populations[p.name].vars["recordSpk"].view, oracle.record(p.name, rows)), f"recording of {p.name} differs"
    assert model.synaptic_event_count == oracle.events() and oracle.events() > 50000
    model.set_step_queue(0)
    model.unload()


def test_plan_can_be_switched_off(monkeypatch):
    monkeypatch.setenv("GENNMI_RESIDENT", "0")
    n, depth = 600, 4
    net = Net(name="resident_off", dt=1.0, steps=0)
    net.pops.append(_pop("A", n, 0.6, -60.0 + 9.5 * rng.uniform(7, 1, 0, n)))
    net.syns.append(_projection("AA", "A", "A", n, n, 48, 0.04, 31, depth, 0.4))
    net.steps = 120

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)

    model, oracle, spikes = _run_chunks(net, (120,), check, resident=False)
    model.unload()


@pytest.mark.parametrize("resident", ["1", "0"])
def test_expired_wait_is_reported_not_hung(resident, monkeypatch):
    """Failure path, forced from the host: with a wait bound of zero polls the first word (resident plan) or spike
    count (per-step plans) that has not arrived when it is first looked at makes the work-group raise the device error
    flag and leave; every kernel still ends normally, and the next synchronisation reports the error."""
    from genn_amd import configs
    from genn_amd._abi import GennmiError
    monkeypatch.setenv("GENNMI_SPIN_LIMIT", "0")
    monkeypatch.setenv("GENNMI_RESIDENT", resident)
    net = configs.potjans(neuron_scale=0.05, connectivity_scale=1.0, steps=2000)
    model = model_from_net(net)
    model.load(num_recording_timesteps=2000)
    assert model.runner_info()["resident_plan"] == (resident == "1")
    model.run(2000)
    with pytest.raises(GennmiError, match="bounded wait"):
        model.synchronize()
    model.unload()
    # the bound is per process: restore the default for whatever runs next
    monkeypatch.delenv("GENNMI_SPIN_LIMIT")
    model = model_from_net(net)
    model.load(num_recording_timesteps=100)
    model.run(100)
    model.synchronize()
    model.unload()


@pytest.mark.parametrize("stride,crowded", [(2, 0.0), (5, 0.0), (14, 0.0), (30, 0.5), (30, 1.0), (90, 0.0)])
def test_row_parts_without_delay_inside_their_entries(stride, crowded, monkeypatch):
    """Projections without a ring: a row's part in a tile is up to four synapses in an entry of two quads (stride 2), up to 22 in one of eight (5, 14),
    longer than that (30 targets crowded into one tile, in some or in all rows) or too long for any entry (90).  Weights are pushed between
    launches, so that the entries' copies of them are rebuilt.  (The tile path adds a step's sums, not its weights one by one: the single
    steps in between go without it.)"""
    monkeypatch.setenv("GENNMI_TILE_FLOATS", "0")
    n_a, n_b = 700, 600
    net = Net(name="resident_inline", dt=1.0, steps=0)
    net.pops.append(_pop("A", n_a, 0.62, -60.0 + 9.5 * rng.uniform(5, 1, 0, n_a)))
    net.pops.append(_pop("B", n_b, 0.45, -60.0 + 9.5 * rng.uniform(5, 2, 0, n_b)))
    ab = _projection("AB", "A", "B", n_a, n_b, stride, 3.0 / stride, 21)
    rows = rng.uniform(5, 3, 0, n_a) < crowded
    ab.ind[rows] = np.sort(ab.ind[rows] % 250, axis=1)
    ab.row_length[::7] = stride // 2                     # (some rows shorter, one in 49 empty)
    ab.row_length[::49] = 0
    net.syns.append(ab)
    net.syns.append(_projection("BA", "B", "A", n_b, n_a, stride, -2.0 / stride, 22))
    net.steps = 260
    pushed = []

    def check(model, oracle):
        compare_state(net, model, oracle, "after a chunk", exact=True)
        if not pushed:
            pushed.append(True)
            for s in net.syns:
                g = model.synapse_populations[s.name].vars["g"]
                g.view[:] = g.view * np.float32(0.5)
                g.push_to_device()
                oracle.syn_g(s.name)[:] *= np.float32(0.5)
    model, oracle, spikes = _run_chunks(net, [100, -3, 97, 60], check)
    assert spikes > 2000
    model.unload()


@pytest.mark.parametrize("n_c, targets, quads", [(None, 0, 8), (20, 5, 8), (100, 60, 4)])
def test_one_projection_does_not_set_every_entry(n_c, targets, quads, monkeypatch):
    """Two populations whose row parts want entries of eight quads (14 targets over 2.3 tiles: 6 a part).  A third one smaller than a tile has the
    whole of a row, 5 targets, in its only part, which asks for no more than the others; parts of 60 are too long for any entry: four quads."""
    monkeypatch.setenv("GENNMI_TILE_FLOATS", "0")
    n_a, n_b = 700, 600
    net = Net(name="resident_entries", dt=1.0, steps=120)
    net.pops.append(_pop("A", n_a, 0.62, -60.0 + 9.5 * rng.uniform(5, 1, 0, n_a)))
    net.pops.append(_pop("B", n_b, 0.45, -60.0 + 9.5 * rng.uniform(5, 2, 0, n_b)))
    net.syns.append(_projection("AB", "A", "B", n_a, n_b, 14, 0.2, 21))
    net.syns.append(_projection("BA", "B", "A", n_b, n_a, 14, -0.15, 22))
    if n_c:
        net.pops.append(_pop("C", n_c, 0.3, -60.0 + 9.5 * rng.uniform(5, 3, 0, n_c)))
        net.syns.append(_projection("AC", "A", "C", n_a, n_c, targets, 0.01, 23))

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)

    model, oracle, spikes = _run_chunks(net, (60, 60), check)
    info = model.runner_info()
    assert (info["resident_tile"], info["resident_quads"], info["resident_walkers"]) == (256, quads, False)
    assert spikes > 700
    model.unload()


@pytest.mark.parametrize("n_a, n_b, depth, models, poisson", [
    (256, 1, 0, 1, False), (250, 255, 1, 1, False), (32760, 3, 0, 1, False), (32760, 260, 2, 1, False),            # few tiles, threads share a tile's word
    (65000, 300, 3, 2, False), (65500, 200, 5, 1, True), (65530, 300, 0, 2, True), (65530, 300, 4, 2, False),      # up to, and one beyond, 256 tiles of 256
    (130000, 1000, 3, 1, False), (130800, 500, 2, 1, True), (130800, 500, 0, 1, False),                           # tiles of 512 and 1024
    (2000, 300, 0, 1, True), (9000, 300, 0, 1, False), (9000, 300, 0, 1, True), (9000, 300, 0, 2, False),          # entries of all sizes
    (5000, 700, 0, 3, False), (5000, 700, 6, 3, False), (70000, 700, 3, 3, True), (131000, 600, 0, 3, False)])     # more than two postsynaptic models
def test_every_number_of_tiles(n_a, n_b, depth, models, poisson, monkeypatch):
    """Which of the kernel's instances runs depends on how many neurons a tile needs (256, 320, 512 or 1024 for a tile a compute unit), rings,
    postsynaptic models a population and sources; a ring of one slot is a case of its own (everything is due at once).  Every (target, postsynaptic model) has one projection: identical.
    (The tile path adds a step's sums, not its weights one by one: the single steps in between go without it.)"""
    monkeypatch.setenv("GENNMI_TILE_FLOATS", "0")
    net = Net(name="resident_tiles", dt=1.0, steps=0)
    net.pops.append(_pop("A", n_a, 0.62, -60.0 + 9.9 * rng.uniform(5, 1, 0, n_a)))
    net.pops.append(_pop("B", n_b, 0.45, -60.0 + 9.9 * rng.uniform(5, 2, 0, n_b)))
    if poisson:
        net.css.append(CurrentSource("A_bg", "poisson_exp", "A", params=dict(weight=0.2, tauSyn=2.0, rate=800.0)))
    def ring(k):
        return dict(depth=depth, due_share=0.3) if depth > 1 else dict(depth=0)
    for k in range(models):
        net.syns.append(_projection(f"BA{k}", "B", "A", n_b, n_a, 40, 0.21 / (k + 1), 11 + k, tau=5.0 + k, **ring(k)))
    net.syns.append(_projection("AB", "A", "B", n_a, n_b, 4, 0.002, 31, **ring(0)))
    if depth == 1:
        for s in net.syns:
            s.wum, s.d, s.max_den_delay = "static_delay", np.zeros(s.ind.shape, np.uint8), 1
    net.steps = 30

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)

    model, oracle, spikes = _run_chunks(net, (14, -2, 14), check)
    assert spikes > n_a // 16
    model.unload()


@pytest.mark.parametrize("sizes, targets, depth, models, poisson, chosen", [
    ((4000,), 80, 0, 1, False, (256, 8, False)), ((8000, 400), 20, 0, 1, False, (256, 8, False)), ((8000, 400), 60, 0, 1, False, (256, 4, False)),
    ((8000, 400), 20, 0, 1, True, (256, 4, False)), ((20000,), 100, 0, 1, False, (256, 4, False)), ((60000,), 80, 0, 1, False, (256, 2, False)),
    ((100000,), 80, 0, 1, False, (512, 2, False)), ((70000,), 150, 0, 1, False, (512, 4, False)), ((70000,), 8, 0, 3, False, (512, 4, False)),
    ((250000,), 20, 0, 1, False, (1024, 2, False)), ((200000, 3000), 10, 0, 1, False, (1024, 4, False)), ((250000,), 20, 0, 1, True, (1024, 4, False)),
    ((40000,), 20, 5, 1, False, (256, 4, True)), ((78000,), 8, 5, 1, False, (320, 4, True)), ((78000,), 8, 35, 2, True, (320, 4, True)),
    ((78000,), 8, 5, 3, False, (512, 4, False)), ((120000,), 8, 5, 2, True, (512, 4, True)), ((240000,), 8, 5, 1, False, (1024, 2, False)),
    ((6200,) * 40, 2, 0, 1, False, (0, 0, False)), ((2000,) * 40, 2, 0, 1, False, (512, 2, False))])
def test_tiles_and_entries_by_rule(sizes, targets, depth, models, poisson, chosen):
    """Which tile, entry and walkers a network gets: the smallest tile with a compute unit for each and room for the rings (tiles of 320 have
    walkers only), entries by the due synapses of a row part where there are instances to choose from.  40 populations of 6,200 are 280 tiles
    of 1,024 and step with the other plans."""
    net = Net(name="resident_rule", dt=1.0, steps=8)
    for p, n in enumerate(sizes):
        net.pops.append(_pop(f"P{p}", n, 0.62, np.full(n, -60.0)))
        if poisson and p == 0:
            net.css.append(CurrentSource("bg", "poisson_exp", "P0", params=dict(weight=0.2, tauSyn=2.0, rate=800.0)))
        for k in range(models):
            net.syns.append(_projection(f"S{p}_{k}", f"P{(p + 1) % len(sizes)}", f"P{p}", sizes[(p + 1) % len(sizes)], n, targets, 0.01, 11 + k, depth, 0.2, tau=5.0 + k))
    model = model_from_net(net)
    model.load(num_recording_timesteps=net.steps)
    info = model.runner_info()
    assert (info["resident_tile"], info["resident_quads"], info["resident_walkers"]) == chosen
    model.unload()


@pytest.mark.parametrize("tile, quads, rings, models, poisson, tiles", [
    (256, 4, "all", 2, False, 3), (256, 4, "all", 1, True, 3), (320, 4, "all", 2, False, 3), (320, 4, "all", 2, True, 3),             # walkers
    (512, 4, "all", 2, False, 3), (512, 4, "all", 2, True, 3),
    (256, 2, "none", 2, False, 3), (256, 2, "some", 2, False, 130), (256, 4, "none", 2, False, 3), (256, 4, "some", 2, True, 3),
    (256, 8, "none", 2, False, 3), (256, 8, "none", 2, False, 31), (256, 8, "none", 2, False, 33), (256, 8, "some", 2, False, 3),      # eight lanes an entry, or one
    (512, 2, "none", 2, False, 3), (512, 2, "some", 1, False, 3), (512, 4, "none", 2, False, 3), (512, 4, "some", 2, False, 3), (512, 4, "none", 2, True, 3),
    (1024, 2, "none", 2, False, 3), (1024, 2, "all", 2, False, 3), (1024, 4, "none", 1, False, 3), (1024, 4, "all", 2, False, 3), (1024, 4, "some", 2, True, 3),
    (256, 4, "all", 3, False, 3), (512, 4, "some", 3, True, 3), (1024, 2, "none", 3, False, 3)])                                       # any number of postsynaptic models
def test_every_instance(tile, quads, rings, models, poisson, tiles, monkeypatch):
    """Every instance of the kernel, tile and entry size given by environment.  Row parts between none and forty synapses: inside entries of any
    size or too long for them."""
    monkeypatch.setenv("GENNMI_TILE_FLOATS", "0")
    monkeypatch.setenv("GENNMI_RESIDENT_TILE", str(tile))
    monkeypatch.setenv("GENNMI_RESIDENT_QUADS", str(quads))
    n_a, n_b, depth = tiles * tile - 5, 200, 5
    net = Net(name="resident_instance", dt=1.0, steps=30)
    net.pops.append(_pop("A", n_a, 0.62, -60.0 + 9.9 * rng.uniform(5, 1, 0, n_a)))
    net.pops.append(_pop("B", n_b, 0.45, -60.0 + 9.9 * rng.uniform(5, 2, 0, n_b)))
    if poisson:
        net.css.append(CurrentSource("A_bg", "poisson_exp", "A", params=dict(weight=0.2, tauSyn=2.0, rate=800.0)))
    def ring(k):
        return dict(depth=depth, due_share=0.3) if rings == "all" or (rings == "some" and k == 0) else dict(depth=0)
    for k in range(models):
        net.syns.append(_projection(f"BA{k}", "B", "A", n_b, n_a, (40, 8, 16)[k], 0.21 / (k + 1), 11 + k, tau=5.0 + k, **ring(k)))
    net.syns.append(_projection("AB", "A", "B", n_a, n_b, 40, 0.002, 31, **ring(models)))
    net.syns.append(_projection("BB", "B", "B", n_b, n_b, 6, 0.02, 32, tau=9.0, **ring(models)))
    for s in net.syns:
        s.row_length[::7] = s.row_stride // 2
        s.row_length[::49] = 0

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)

    model, oracle, spikes = _run_chunks(net, (14, -2, 14), check)
    info = model.runner_info()
    assert (info["resident_tile"], info["resident_quads"], info["resident_walkers"]) == (tile, quads, rings == "all" and models <= 2 and tile <= 512)
    assert spikes > n_a // 16
    model.unload()


@pytest.mark.parametrize("together", [1, 3, 4, 5, 8, 33, 256])
@pytest.mark.parametrize("depth", [0, 5])
def test_spikes_of_one_tile_in_one_step(together, depth):
    """Of a tile of 256 neurons `together` fire in the first step: up to three travel in the tile's word and more in its side list, and the
    128 threads that watch the tile of so small a network take one, some or none of them each."""
    n_a, n_b = 256, 200
    net = Net(name="resident_together", dt=1.0, steps=40)
    net.pops.append(_pop("A", n_a, 0.62, np.where(np.arange(n_a) * 97 % 256 < together, -50.01, -60.0)))
    net.pops.append(_pop("B", n_b, 0.3, np.full(n_b, -58.0)))
    net.pops[0].params["Ioffset"] = 0.55
    net.syns.append(_projection("AB", "A", "B", n_a, n_b, 20, 0.3, 21, depth, 0.3))
    net.syns.append(_projection("AA", "A", "A", n_a, n_a, 9, 0.2, 22, depth, 0.3))

    def check(model, oracle):
        compare_state(net, model, oracle, f"after {model.timestep} steps", exact=True)

    model, oracle, spikes = _run_chunks(net, (6, 34), check)
    assert int(np.unpackbits(oracle.record("A", 40).reshape(40, -1)[0].view(np.uint8)).sum()) == together
    model.unload()


@pytest.mark.parametrize("threads", [False, True])
def test_networks_that_do_not_fit_together(threads):
    """Two networks of 158 tiles, each a compute unit's worth, do not fit on the chip together, and a third of 13 fits beside one of them.
    Stepped at the same time, a launch behind the other's without a wait between them or from a thread each, every one is as if alone."""
    steps, chunk = 48, 4
    sizes = (40000, 40000, 3000)
    nets = []
    for k, n in enumerate(sizes):
        net = Net(name=f"resident_beside{k}", dt=1.0, steps=steps)
        net.pops.append(_pop("A", n, 0.62, -60.0 + 9.9 * rng.uniform(5, 1 + k, 0, n)))
        net.pops.append(_pop("B", 300, 0.45, -60.0 + 9.9 * rng.uniform(6, 1 + k, 0, 300)))
        net.syns.append(_projection("AB", "A", "B", n, 300, 4, 0.002, 31 + k, 4, 0.3))
        net.syns.append(_projection("BA", "B", "A", 300, n, 40, 0.2, 41 + k, 4, 0.3))
        nets.append(net)
    models = [model_from_net(net) for net in nets]
    for model, n in zip(models, sizes):
        model.load(num_recording_timesteps=steps)
        info = model.runner_info()
        assert info["resident_plan"] and info["resident_tile"] == 256 and info["resident_walkers"]
    if threads:
        failed = []

        def work(model):
            try:
                for _ in range(steps // chunk):
                    model.run(chunk)
                model.synchronize()
            except Exception as e:
                failed.append(e)

        workers = [threading.Thread(target=work, args=(model,)) for model in models]
        for w in workers:
            w.start()
        for w in workers:
            w.join()
        assert not failed
    else:
        for _ in range(steps // chunk):
            for model in models:
                model.run(chunk)
        for model in models:
            model.synchronize()
    for net, model in zip(nets, models):
        oracle = OracleNet(net, num_recording_timesteps=steps)
        oracle.run(steps)
        compare_state(net, model, oracle, f"of {net.name}", exact=True)
        model.pull_recording_buffers_from_device()
        for p in net.pops:
            assert np.array_equal(model.neuron_populations[p.name].vars["recordSpk"].view, oracle.record(p.name, steps)), f"recording of {p.name} differs"
        assert model.synaptic_event_count == oracle.events() > 0
        model.unload()


def test_no_room_for_the_tables_means_another_plan(monkeypatch):
    """A network whose segment tables take 2 GB a projection, on a card with 3 GiB free: the second table finds no room, the first goes back, and
    the network steps with the other plans."""
    monkeypatch.setenv("GENNMI_TILE_FLOATS", "0")
    n, gib = 250000, 1 << 30
    net = Net(name="resident_no_room", dt=1.0, steps=12)
    net.pops.append(_pop("A", n, 0.62, -60.0 + 9.9 * rng.uniform(5, 1, 0, n)))
    for k in range(2):
        net.syns.append(_projection(f"AA{k}", "A", "A", n, n, 2, 0.1, 11 + k, tau=5.0 + k))
    model = model_from_net(net)
    release_cached_memory()
    free, _ = torch.cuda.mem_get_info()
    taken = C.c_void_p()
    _abi.check(_abi.load().gennmi_malloc(C.byref(taken), free - 3 * gib))
    try:
        model.load(num_recording_timesteps=net.steps)
        assert not model.runner_info()["resident_plan"]
        release_cached_memory()
        assert torch.cuda.mem_get_info()[0] > 2.5 * gib
    finally:
        _abi.check(_abi.load().gennmi_free(taken))
        release_cached_memory()
    oracle = OracleNet(net, num_recording_timesteps=net.steps)
    model.run(net.steps)
    oracle.run(net.steps)
    model.synchronize()
    compare_state(net, model, oracle, "with the other plans", exact=True)
    assert model.synaptic_event_count == oracle.events() > 0
    model.unload()
