"""Decoding of spike recordings (host code of the device library; no device calls)."""
import ctypes as C

import numpy as np
import pytest

from genn_amd import _abi
from genn_amd.genn_model import GeNNModel


@pytest.mark.parametrize("num_neurons", [1, 31, 32, 33, 64, 100])
@pytest.mark.parametrize("batch", [1, 3])
def test_recording_decodes_to_the_bits_that_are_set(num_neurons, batch):
    """Every bit is one (time, neuron) pair, rows in time order and neurons ascending; bits beyond the population are ignored."""
    steps, words = 7, (num_neurons + 31) // 32
    rec = np.random.default_rng(num_neurons * 10 + batch).integers(0, 1 << 32, (steps, batch, words), dtype=np.uint32)
    rec[3] = 0
    model = GeNNModel("float", "decode", batch_size=batch, dt=0.1)
    pop = model.add_neuron_population("P", num_neurons, "LIF")
    model.num_recording_timesteps, model.timestep = steps, 19
    pop.vars["recordSpk"] = type("Buffer", (), {"view": rec.reshape(-1)})()
    bits = np.unpackbits(rec.view(np.uint8), axis=2, bitorder="little")[:, :, :num_neurons]
    for b, (times, ids) in enumerate(pop.spike_recording_data):
        step, neuron = np.nonzero(bits[:, b])
        assert times.dtype == np.float64 and ids.dtype == np.uint32
        assert np.array_equal(ids, neuron) and np.array_equal(times, (12 + step) * 0.1)


def test_decoding_refuses_arrays_that_are_too_short():
    rec, count = np.array([7], np.uint32), C.c_size_t(2)
    times, ids = np.empty(2), np.empty(2, np.uint32)
    rc = _abi.load().gennmi_decode_recording(rec.ctypes.data, 1, 1, 32, 0.0, 1.0, times.ctypes.data, ids.ctypes.data, C.byref(count))
    assert rc != 0
