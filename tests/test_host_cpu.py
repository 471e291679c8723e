"""CPU tests of the host side and of the C-ABI library's surface (no device calls)."""
import ctypes as C
import math
import os
import re
import subprocess

import numpy as np
import pytest
import torch

from genn_amd import _abi, configs, netgen, rng
from genn_amd.genn_model import GeNNModel, init_postsynaptic, init_weight_update, lit32, field32, model_from_net

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "genn_mi355x.h")).read()
    declared = set(re.findall(r"\b(gennmi_[a-z0-9_]+)\s*\(", header))
    assert declared, "no prototypes found in the header"
    lib = _abi.load()
    for name in declared:
        assert hasattr(lib, name), f"{name} is declared in include/genn_mi355x.h but not exported"
    assert declared == set(_abi.SYMBOLS), "ctypes prototype table and header disagree"


def test_struct_layout_matches_the_library():
    sizes = (C.c_size_t * 5)()
    assert _abi.load().gennmi_abi_struct_sizes(C.byref(sizes)) == 0
    assert list(sizes) == [C.sizeof(_abi.Psm), C.sizeof(_abi.Cs), C.sizeof(_abi.NeuronUpdateGroup),
                           C.sizeof(_abi.PresynapticUpdateGroup), C.sizeof(_abi.PostsynapticUpdateGroup)]


def test_error_reporting_without_a_device():
    lib = _abi.load()
    assert lib.gennmi_abi_struct_sizes(None) == -2
    assert b"null" in lib.gennmi_last_error()
    with pytest.raises(_abi.GennmiError):
        _abi.check(lib.gennmi_runner_finalise(None))


def test_literal_and_field_rounding():
    # 0.1 as a literal and as a struct field agree; a value next to a rounding boundary does not
    assert lit32(0.1) == field32(0.1) == np.float32(0.1)
    x = float(np.float32(1.0)) + 2.0 ** -24 + 2.0 ** -40     # just above the midpoint of two floats
    assert field32(x) == np.nextafter(np.float32(1.0), np.float32(2.0))
    assert lit32(x) == np.float32(float("%.9e" % x))
    assert lit32(math.exp(-0.1 / 20.0)) == np.float32("9.950124792e-01")
    assert lit32(0.0) == 0.0 and lit32(-65.0) == np.float32(-65.0)


def test_literals_are_of_values_not_of_objects():
    """An array of one value is a value, one that is written again is another, and zero has two signs."""
    for x in (np.array(0.1), np.array([0.1]), np.float32(0.1), 0.1):
        assert lit32(x) == np.float32(float("%.9e" % float(np.asarray(x).reshape(-1)[0])))
    held = torch.tensor(1.5, dtype=torch.float64)
    assert lit32(held) == np.float32(1.5)
    held.fill_(2.5)
    assert lit32(held) == np.float32(2.5)
    assert [np.signbit(lit32(z)) for z in (0.0, -0.0, 0.0)] == [False, True, False]
    assert np.isnan(lit32(float("nan"))) and lit32(-np.inf) == -np.inf


def test_generators_agree_and_shapes_hold():
    assert np.array_equal(netgen.words(9, 3, 17, 500), rng.words(9, 3, 17, 500))
    assert np.array_equal(netgen.normal_f32(9, 3, 0, 500, 1.0, 2.0), (1.0 + 2.0 * rng.normal(9, 3, 0, 500)).astype(np.float32))
    rl, ind = netgen.fixed_probability(2, 5, 300, 200, 0.1, pad=4)
    assert ind.shape[1] % 4 == 0 and ind.shape[1] >= rl.max()
    assert abs(rl.mean() - 20.0) < 1.5
    for r in range(300):
        row = ind[r, :rl[r]].astype(np.int64)
        assert np.all(np.diff(row) > 0) and (len(row) == 0 or row[-1] < 200)
    rl, ind = netgen.fixed_number_total(2, 6, 50, 40, 1000)
    assert rl.sum() == 1000
    for r in range(50):
        assert np.all(np.diff(ind[r, :rl[r]].astype(np.int64)) >= 0)       # multapses allowed
    rl, ind = netgen.fixed_number_post(2, 7, 10, 1000, 64)
    assert np.all(rl == 64) and ind.shape == (10, 64)
    d = netgen.rows_clipped_normal_delay(2, 8, rl, 64, 15.0, 7.5, 0.0, 42.89)
    assert d.min() >= 0 and d.max() <= 43


def test_full_scale_microcircuit_counts():
    """298,624,465 synapses in 54 non-empty projections, 43 delay slots (userproject/potjans_microcircuit.py:108-133, 181-190)."""
    pops = [l + p for l in configs.PD_LAYERS for p in ("E", "I")]
    total, nonempty = 0, 0
    for trg in pops:
        for src in pops:
            k = int(round(configs.pd_full_num_inputs(src, trg) * float(configs.PD_NUM[trg])))
            total += k
            nonempty += k > 0
    assert total == 298624465 and nonempty == 54
    assert sum(configs.PD_NUM.values()) == 77169
    max_delay = configs.PD_MEAN_DELAY["E"] + configs.PD_DELAY_SD["E"] * configs.PD_NORM_Q9999
    assert int(round(max_delay / 0.1)) == 43


def test_postsynaptic_fusing_and_child_order():
    """Fusing walks incoming projections last-to-first (src/genn/genn/neuronGroup.cc:41-96): the owner of a fused
    outPost is the LAST projection added, and unfused children keep reverse creation order."""
    net = configs.potjans(neuron_scale=0.01, connectivity_scale=0.05, steps=10)
    m = model_from_net(net)
    for n in m.neuron_populations.values():
        assert len(n.fused_psm) == 1
        assert n.fused_psm[0][0] is n.in_syn[-1]
        assert all(s.fused_ps_target is n.in_syn[-1] for s in n.in_syn)
    net = configs.vogels_abbott(n=100, steps=10, p=0.1)
    m = model_from_net(net)
    e = m.neuron_populations["E"]
    assert [grp[0].name for grp in e.fused_psm] == ["IE", "EE"]


def test_unsupported_models_fail_loudly():
    m = GeNNModel("float", "x")
    with pytest.raises(NotImplementedError):
        m.add_neuron_population("p", 10, "TraubMiles", {}, {})
    with pytest.raises(NotImplementedError):
        init_weight_update("PiecewiseSTDP")
    with pytest.raises(NotImplementedError):
        init_postsynaptic("ExpCond")
    with pytest.raises(NotImplementedError):
        GeNNModel("double", "x")
    p = m.add_neuron_population("p", 10, "LIF", {}, {})
    with pytest.raises(RuntimeError):
        m.load()           # build() first, as in the reference


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode != 0 and "one GPU" in (r.stderr + r.stdout)


def test_philox_known_answers():
    """The generator under the on-device initialisation snippets, through the library's host entry point and the numpy
    restatement the GPU tests compare device output with: both must give the published known-answer vectors."""
    import ctypes as C
    from philox_ref import KNOWN_ANSWERS, philox4x32
    lib = _abi.load()
    for counter, key, want in KNOWN_ANSWERS:
        out = (C.c_uint32 * 4)()
        assert lib.gennmi_philox4x32(C.byref((C.c_uint32 * 4)(*counter)), C.byref((C.c_uint32 * 2)(*key)), C.byref(out)) == 0
        assert tuple(out) == want
        assert tuple(int(w) for w in philox4x32(*counter, *key)) == want


def test_max_row_length_follows_the_snippets():
    """Row strides of the built-in connectivity snippets against the known answers of the reference's unit test for
    binomialInverseCDF (tests/unit/binomial.cc:15-35: square matrices of 1, 1000 and 10^6 neurons at three probabilities)."""
    from genn_amd.genn_model import max_row_length
    table = {0.02: (1, 47, 20897), 0.1: (1, 153, 101914), 1.0: (1, 1000, 1000000)}
    for prob, want in table.items():
        for size, stride in zip((1, 1000, 1000000), want):
            assert max_row_length("FixedProbability", {"prob": prob}, size, size) == stride
    assert max_row_length("FixedNumberPostWithReplacement", {"num": 37}, 100, 100) == 37
    assert max_row_length("OneToOne", {}, 100, 100) == 1


def test_lists_of_a_convolution_cost_no_work_group(tmp_path):
    """A layer of a feed-forward network lists its steps' inputs in LDS only where as many work-groups stay on a compute unit as without the lists, or as the
    launch has: four by their registers, and by 160 KiB of LDS in parts of 1,280 bytes.  Which layers are taken, and their rows, do not depend on the lists."""
    (tmp_path / "layout.cc").write_text("""#include "genn_mi355x_ahead_layout.h"
extern "C" void layout(const int *c, unsigned batch, unsigned units, unsigned long long *out)
{
    const AheadConvLayout l = aheadConvLayout(c[0], c[1], c[2], c[3], c[4], c[5], batch, units);
    out[0] = l.fits; out[1] = l.rowsPerBlock; out[2] = l.listDepth; out[3] = l.bytes;
}
""")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "genn_amd", "csrc"), "-o", str(tmp_path / "layout.so"), str(tmp_path / "layout.cc")], check=True)
    layout = C.CDLL(str(tmp_path / "layout.so")).layout

    def resident(size):
        return min(4, 163840 // (-(-(size + 288) // 1280) * 1280))

    units, listed, shallower = 256, 0, 0
    shapes = [(64, w, 8, 32, 5, 16) for w in range(36, 44)] + [(64, 72, 16, 32, 3, 16), (16, 16, 9, 32, 5, 16), (64, 64, 1, 32, 3, 16), (64, 64, 16, 32, 3, 16)]
    shapes += [(h, w, ic, oc, k, b) for h, w in ((5, 7), (33, 47), (64, 64), (200, 31)) for ic in (1, 2, 3, 5, 8, 13, 16, 20, 40, 60) for oc, b in ((1, 1), (33, 2), (64, 16), (1056, 3)) for k in (1, 3, 5)]
    for h, w, ic, oc, k, b in shapes:
        out = (C.c_ulonglong * 4)()
        layout((C.c_int * 6)(k, k, ic, h, w, oc), b, units, out)
        fits, rows, depth, size = out
        inputs, columns = k * k * ic, b * (-(-oc // 32))
        bare = lambda r: 4 * ((r + k - 1) * (w - 1 + k) * ic + 32 * inputs + (inputs + 1) // 2 + 8 * (inputs + 1))
        most = max(1, min(h, h * columns // (4 * units)))
        while bare(most) > 65536 and most > 1:
            most -= 1
        assert (bool(fits), rows) == (bare(most) <= 83968, most), (h, w, ic, oc, k, b)
        if not fits:
            continue
        needed = -(-(-(-h // rows) * columns) // units)
        assert resident(size) >= min(needed, resident(bare(rows))), (h, w, ic, oc, k, b, depth, size)
        assert depth % 4 == 0 and depth <= min(16, inputs // 16 * 4) and (depth or size == bare(rows)) and size >= 4 * 128 * depth and inputs * 128 < 65536
        listed, shallower = listed + (depth != 0), shallower + (depth < min(16, inputs // 16 * 4))
    assert listed > 100 and shallower > 5


def test_counters_are_attached_to_the_code_they_were_read_on(tmp_path, monkeypatch):
    """The benchmark's figures of hardware counters go with every file that their kernel's code comes from: the convolution's step has its neurons' update
    and its products from the other kernel files."""
    import shutil
    import bench
    files = {key: measured["kernel_source"][0] for key, measured in bench.MEASURED_TRAFFIC_BYTES.items()}
    assert {"conv_step_kernels", "neuron_kernels", "synapse_kernels", "device"} <= set(files["conv", 1000, 100])
    assert {"resident_kernels", "device"} <= set(files["potjans", 20, 5])
    shutil.copytree(os.path.join(ROOT, "genn_amd", "csrc"), tmp_path / "genn_amd" / "csrc")
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    for names in files.values():
        seen = [bench.source_digest(names)]
        for name in names:
            with open(tmp_path / "genn_amd" / "csrc" / f"genn_mi355x_{name}.h", "a") as f:
                f.write("//")
            seen.append(bench.source_digest(names))
        assert len(set(seen)) == len(names) + 1
