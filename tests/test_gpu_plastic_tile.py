"""The tile path of plastic projections with the presynaptic-spike rule's share worked out once per target in LDS
(GENNMI_TILE_FACTORS: 0 never, 1 by the rule, 2 in every step that takes the tile path): the same operations on the same numbers, so
weights must be the same bit for bit wherever the spikes are, and spikes those of the CPU oracle."""
import numpy as np
import pytest

from genn_amd import configs
from genn_amd.genn_model import model_from_net
from oracle.genn_cpu import OracleNet

pytestmark = pytest.mark.gpu


# tiles: all targets in one; 9 of them with a remainder; one of 32 targets, the smallest with room for its bits
@pytest.mark.parametrize("rule", ["stdp_trace", "stdp_additive"])
@pytest.mark.parametrize("tile_floats,n", [("16384", 2500), ("512", 2501), ("66", 300)])
def test_weights_are_the_same_with_and_without(rule, tile_floats, n, monkeypatch):
    monkeypatch.setenv("GENNMI_TILE_FLOATS", tile_floats)
    monkeypatch.setenv("GENNMI_TILE_THREADS", "512")
    steps = 60
    # strong drive: bursts in which sources and targets of a synapse fire together, so both rules meet on it
    net = configs.plastic_stdp(n=n, n_src=100, steps=steps, fan=n // 10, src_fan=50, src_w=6.0, ioffset=0.6, rule=rule)
    ee = next(s for s in net.syns if s.name == "EE")
    ee.g = np.array(ee.g)
    ee.g[::5] = 1.75             # beyond wMax: a synapse that neither rule touches keeps it, one that is touched is clipped
    got = []
    for factors in ("0", "1", "2"):
        monkeypatch.setenv("GENNMI_TILE_FACTORS", factors)
        model = model_from_net(net)
        model.load(num_recording_timesteps=steps)
        for _ in range(steps):
            model.step_time()
        model.pull_recording_buffers_from_device()
        got.append((model.synapse_populations["EE"].vars["g"].pull_from_device().copy(), {p.name: model.neuron_populations[p.name].vars["recordSpk"].view.copy() for p in net.pops}))
        col_stride = model.synapse_populations["EE"].col_stride
        model.unload()
    oracle = OracleNet(net, num_recording_timesteps=steps, col_stride={"EE": col_stride})
    oracle.run(steps)
    spikes = 0
    for p in net.pops:
        want = oracle.record(p.name, steps)
        for g, raster in got:
            assert np.array_equal(raster[p.name].reshape(-1), want.reshape(-1)), p.name
        spikes += int(np.unpackbits(want.view(np.uint8)).sum())
    assert spikes > 2 * n
    valid = (np.arange(ee.ind.shape[1])[None, :] < np.asarray(ee.row_length)[:, None]).reshape(-1)
    want = oracle.syn_g("EE").reshape(-1)[valid]
    for g, raster in got:
        assert np.array_equal(g.reshape(-1)[valid], got[0][0].reshape(-1)[valid])
        assert np.abs(g.reshape(-1)[valid] - want).max() <= 1e-5
    assert (np.abs(want - np.asarray(ee.g).reshape(-1)[valid]) > 1e-3).mean() > 0.5


def test_short_rows_are_walked_about_as_fast_as_long_ones():
    """A burst of the targets walks every row.  Three million synapses in rows of 30 took 10 times as long as in rows of 300 when a wavefront looked at
    rows far apart and took two of them at a time, whatever their length."""
    from genn_amd.genn_model import GeNNModel, init_postsynaptic, init_sparse_connectivity, init_var, init_weight_update
    m, took = 1000, {}
    lif = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, TauRefrac=5.0)
    rule = dict(tauPlus=20.0, tauMinus=20.0, aPlus=1e-6, aMinus=1e-6, wMin=0.0, wMax=1.0)
    for n, fan in ((100000, 30), (10000, 300)):
        model = GeNNModel("float", "rows", dt=0.5)
        model.seed, model.timing_enabled = 7, True
        a = model.add_neuron_population("A", n, "LIF", dict(lif, Ioffset=0.0), {"V": -60.0, "RefracTime": 0.0})
        b = model.add_neuron_population("B", m, "LIF", dict(lif, Ioffset=4.0), {"V": init_var("Uniform", {"min": -60.0, "max": -50.0}), "RefracTime": 0.0})
        model.add_synapse_population("AB", "SPARSE", a, b, init_weight_update("STDPTrace", rule, {"g": init_var("Uniform", {"min": 0.0, "max": 0.5})}, {"preTrace": 0.0}, {"postTrace": 0.0}),
                                     init_postsynaptic("ExpCurr", {"tau": 5.0}), init_sparse_connectivity("FixedNumberPostWithReplacement", {"num": fan}))
        model.build()
        model.load()
        rounds = []
        for _ in range(5):
            before = model.postsynaptic_update_time
            for _ in range(40):
                model.step_time()
            rounds.append(model.postsynaptic_update_time - before)
        took[n] = min(rounds)
        model.unload()
    assert 0.0 < took[100000] < 4.0 * took[10000], took


def test_bursts_of_short_rows_do_not_depend_on_how_many_work_groups_a_tile_gets():
    """Rows of 9 synapses over 40 tiles share cache lines between the tiles' work-groups.  Dealt out tile by tile, those of one line met in one L2 only where a
    tile had a multiple of 8 or 4 of them: a step of 720,000 neurons (17 to a tile) took 1.5 times as long as one of 650,000 (20), now 1.1 times."""
    from genn_amd.genn_model import GeNNModel, init_postsynaptic, init_sparse_connectivity, init_var, init_weight_update
    lif, took = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=4.0, TauRefrac=2.0), {}
    for n in (650000, 720000):
        model = GeNNModel("float", "burst", dt=1.0)
        model.seed, model.timing_enabled = 11, True
        size = {"E": n * 4 // 5, "I": n // 5}
        pops = {k: model.add_neuron_population(k, size[k], "LIF", lif, {"V": init_var("Uniform", {"min": -60.0, "max": -50.0}), "RefracTime": 0.0}) for k in "EI"}
        for src in "EI":
            for trg, num in (("E", 7), ("I", 2)):
                model.add_synapse_population(src + trg, "SPARSE", pops[src], pops[trg], init_weight_update("StaticPulse", {}, {"g": init_var("Uniform", {"min": 0.0, "max": 1e-4})}),
                                             init_postsynaptic("DeltaCurr"), init_sparse_connectivity("FixedNumberPostWithReplacement", {"num": num}))
        model.build()
        model.load()
        rounds = []
        for _ in range(5):
            before = model.presynaptic_update_time
            for _ in range(20):
                model.step_time()
            rounds.append(model.presynaptic_update_time - before)
        took[n] = min(rounds)
        model.unload()
    assert 0.0 < took[720000] < 1.3 * took[650000], took
