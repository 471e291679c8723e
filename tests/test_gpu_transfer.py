"""Copies in the order of a runner's steps: sizes around the chunks they are cut into, offsets around 16 bytes, spike queues of every length."""
import ctypes as C

import numpy as np
import pytest

from genn_amd import _abi, configs
from genn_amd.genn_model import model_from_net

pytestmark = pytest.mark.gpu
CHUNK = 1 << 20


@pytest.fixture(scope="module")
def model():
    m = model_from_net(configs.vogels_abbott(n=1000, steps=20, p=0.1))
    m.load(num_recording_timesteps=20)
    yield m
    m.unload()


@pytest.mark.parametrize("count, dtype", [(1, np.uint8), (15, np.uint8), (17, np.uint8), (CHUNK + 3, np.uint8), (3, np.float32), (CHUNK // 4 - 1, np.float32),
                                          (CHUNK // 4, np.float32), (CHUNK // 4 + 1, np.float32), (6 * CHUNK // 4 + 5, np.uint32)])
def test_arrays_come_back_as_they_were_sent(model, count, dtype):
    a = model._alloc(count, dtype)
    want = np.random.default_rng(count).integers(0, 256, count * np.dtype(dtype).itemsize, dtype=np.uint8)
    a.view.view(np.uint8)[:] = want
    model.step_time()
    a.push_to_device()
    a.view.view(np.uint8)[:] = 0
    model.step_time()
    assert np.array_equal(a.pull_from_device().view(np.uint8), want)
    if dtype == np.float32:
        b = model._alloc(count, dtype)
        b.copy_on_device(a)
        assert np.array_equal(b.pull_from_device().view(np.uint8), want)


@pytest.mark.parametrize("offset", [1, 7, 15, 16, 17])
@pytest.mark.parametrize("nbytes", [1, 14, 33, CHUNK + 1])
def test_parts_of_arrays(model, offset, nbytes):
    a = model._alloc(CHUNK + 64, np.uint8)
    want = np.random.default_rng(nbytes).integers(1, 256, nbytes, dtype=np.uint8)
    lib = _abi.load()
    _abi.check(lib.gennmi_runner_push(model._runner, a.ptr + offset, want.ctypes.data, nbytes))
    got = np.zeros(nbytes + 2, np.uint8)
    _abi.check(lib.gennmi_runner_pull(model._runner, 1, (C.c_void_p * 1)(got.ctypes.data + 1), (C.c_void_p * 1)(a.ptr + offset), (C.c_size_t * 1)(nbytes)))
    assert got[0] == 0 and got[-1] == 0 and np.array_equal(got[1:-1], want)
    whole = a.pull_from_device()
    assert not whole[:offset].any() and not whole[offset + nbytes:].any()


@pytest.mark.parametrize("n, batch, slots", [(1, 1, 1), (255, 2, 1), (257, 3, 4), (300_000, 1, 1), (70_000, 5, 2)])
def test_spike_queues_of_every_length(model, n, batch, slots):
    """Empty, single, work-group sized, full: also queues longer than the part of a chunk a batch gets."""
    lib, rng = _abi.load(), np.random.default_rng(n)
    runner = C.c_void_p()
    _abi.check(lib.gennmi_runner_create(C.byref(runner), 1.0, batch))
    spk, cnt = model._alloc(batch * slots * n, np.uint32), model._alloc(batch * slots, np.uint32)
    spk.view[:] = rng.integers(0, n, spk.count)
    spk.push_to_device()
    got, counts = np.empty((batch, n), np.uint32), np.empty(batch, np.uint32)
    for length in sorted({0, min(1, n), min(256, n), min(257, n), n // 2, n}):
        cnt.view[:] = length
        cnt.view[-1] = n - length
        cnt.push_to_device()
        for slot in (0, slots - 1):
            got[:] = 0xFFFFFFFF
            _abi.check(lib.gennmi_runner_pull_spikes(runner, cnt.ptr, spk.ptr, n, slots, slot, counts.ctypes.data, got.ctypes.data))
            want_counts = cnt.view.reshape(batch, slots)[:, slot]
            assert np.array_equal(counts, want_counts)
            for b in range(batch):
                assert np.array_equal(got[b, :counts[b]], spk.view.reshape(batch, slots, n)[b, slot, :counts[b]])
                assert np.all(got[b, counts[b]:] == 0xFFFFFFFF)
    _abi.check(lib.gennmi_runner_destroy(runner))


# a quad; a work-group's 1,024 floats, four quads a thread, 256 and 512 work-groups', twice around; ends and beginnings on and off 16 bytes, together and apart
@pytest.mark.parametrize("count", [1, 3, 4, 1025, 4095, 4097, 64 * 1024 + 1, 64 * 4096 + 5, 256 * 4096 + 1, (1 << 22), (1 << 22) + 7, 2 * 512 * 4096 + 4099])
@pytest.mark.parametrize("to, at", [(0, 0), (4, 4), (1, 1), (3, 3), (0, 1), (1, 0), (2, 3)])
def test_copies_on_the_device_touch_what_they_name(model, count, to, at):
    lib = _abi.load()
    a, b = model._alloc(count + 8, np.float32), model._alloc(count + 8, np.float32)
    assert a.ptr % 16 == 0 and b.ptr % 16 == 0
    a.view[:] = np.arange(count + 8)
    a.push_to_device()
    b.view[:] = -1.0
    b.push_to_device()
    _abi.check(lib.gennmi_runner_copy_f32(model._runner, b.ptr + 4 * to, a.ptr + 4 * at, count))
    got = b.pull_from_device()
    assert np.array_equal(got[to:to + count], np.arange(at, at + count, dtype=np.float32))
    assert np.all(got[:to] == -1.0) and np.all(got[to + count:] == -1.0)
    a.free()
    b.free()


def test_copies_off_16_bytes_keep_memory_as_busy(model):
    """A large copy whose two sides begin at different offsets of 16 bytes has no quads; with an element a thread under way, and as few work-groups as
    suffice for quads, it took 3.7 times as long as one that has them."""
    import time
    lib, count = _abi.load(), 64 << 20
    a, b = model._alloc(count + 8, np.float32), model._alloc(count + 8, np.float32)
    took = {}
    for to, at in ((0, 0), (0, 1), (1, 1)):
        rounds = []
        for _ in range(12):
            model.synchronize()
            begin = time.perf_counter()
            _abi.check(lib.gennmi_runner_copy_f32(model._runner, b.ptr + 4 * to, a.ptr + 4 * at, count))
            rounds.append(time.perf_counter() - begin)
        took[to, at] = min(rounds)
    a.free()
    b.free()
    assert max(took.values()) < 2.0 * took[0, 0], took
