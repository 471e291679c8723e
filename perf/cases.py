"""What this framework is asked to do, as cases that can be prepared, run and compared.

A case is one pass of a user's program over a loaded network: step it (one call at a time, a block of steps at once, or a
closed loop that reads the spikes after every step), present a batch of samples to it, or build it on the device.  The
networks are the ones of the repository's configurations, stated with the built-in connectivity and variable snippets so
that their matrices are made on the device; everything random comes from the seed.

Spiking networks are not stationary, so ``work()`` counts the activity that a running network of the family settles to.
"""
import math

import numpy as np
import torch

from genn_amd import configs, netgen
from genn_amd.genn_model import (GeNNModel, init_postsynaptic, init_sparse_connectivity, init_toeplitz_connectivity, init_var,
                                 init_weight_update)

LIF = dict(C=1.0, TauM=20.0, Vrest=-60.0, Vreset=-60.0, Vthresh=-50.0, Ioffset=0.55, TauRefrac=5.0)
IZHIKEVICH = dict(a=0.02, b=0.2, c=-65.0, d=8.0)
STDP_TRACE = dict(tauPlus=20.0, tauMinus=20.0, aPlus=0.01, aMinus=0.012, wMin=0.0, wMax=1.0)
STDP_ADDITIVE = dict(tauPlus=20.0, tauMinus=20.0, Aplus=0.01, Aminus=0.012, Wmin=0.0, Wmax=1.0)


def listed():
    return [
        # A robot or an agent in the loop: every 0.1 ms step of a small balanced network is followed by reading its spikes.
        # Nothing but latency: launches, waits and the host's own work.
        dict(name="closed_loop_4k", family="balanced", neurons=4000, fan=80, drive="closed_loop", steps=1),
        # The first network anybody runs, 0.1 s of it at once, its raster read as times and neuron numbers and counted.
        dict(name="balanced_4k", family="balanced", neurons=4000, fan=80, drive="run", steps=1000, read="spikes"),
        # The usual loop of step_time() calls over a network too large to stay on the chip; odd sizes, rows of about 1000.
        dict(name="balanced_300k_steps", family="balanced", neurons=300007, fan=1000, drive="step", steps=50, read="recording"),
        # The full cortical microcircuit (dendritic delays, constant background), 0.1 s of it at once: the headline network.
        dict(name="microcircuit", family="microcircuit", scale=1.0, poisson=False, drive="run", steps=1000, read="recording"),
        # A reduced microcircuit with its Poisson background, stepped call by call, its raster kept.
        dict(name="microcircuit_35_poisson_steps", family="microcircuit", scale=0.35, poisson=True, drive="step", steps=100, read="recording"),
        # 10^6 neurons with 10^9 stored synapses: the bandwidth case, and the largest.
        dict(name="izhikevich_1m", family="izhikevich", neurons=1000000, fan=1000, matrix="SPARSE", drive="run", steps=20, read="recording"),
        # The same network where the matrix does not fit or is not wanted: every row is generated anew for every spike.
        dict(name="izhikevich_1m_procedural", family="izhikevich", neurons=1000000, fan=1000, matrix="PROCEDURAL", drive="run", steps=20, read="recording"),
        # Learning at scale: 32 million plastic synapses under the trace rule, pairings in both directions.
        dict(name="plastic_100k", family="plastic", neurons=100000, fan=500, rule="STDPTrace", drive="run", steps=100, read="recording"),
        # A learning experiment of ordinary size under the built-in additive rule, stepped call by call; no size is even.
        dict(name="plastic_17k_steps", family="plastic", neurons=17011, fan=300, rule="STDP", drive="step", steps=50, read="recording"),
        # Rate-coded inference through a convolutional layer: a batch of 16 samples, each 50 ms, new input spikes every time.
        dict(name="conv_64x64_batch16", family="conv", height=64, width=64, channels_in=16, channels_out=32, kernel=3, batch=16, steps=50),
        # Rate-coded inference through a fully connected layer, one sample of 100 ms.
        dict(name="dense_8192", family="dense", inputs=8192, outputs=8192, batch=1, steps=100),
        # From a model's description to its first possible step: allocation, connectivity and weights made on the device.
        dict(name="build_100k", family="build", neurons=100000, fan=1000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the family as often as the listed ones have it, sizes over the range between and below them."""
    family = rng.choice(["balanced"] * 3 + ["microcircuit"] * 2 + ["izhikevich"] * 2 + ["plastic"] * 2 + ["conv", "dense", "build"])
    drive = rng.choice(["run", "step"])
    if family == "balanced":
        n = _log(rng, 1000, 300000)
        case = dict(family=family, neurons=n, fan=_log(rng, 80, min(1000, n // 4)), drive=rng.choice(["run", "step", "closed_loop"]))
        if case["drive"] == "closed_loop":
            return dict(case, steps=_log(rng, 1, 10))
        case["steps"] = _log(rng, 20, min(1000, 15000000 // n))
        return dict(case, read="spikes" if n * case["steps"] < 4000000 else "recording")
    if family == "microcircuit":
        return dict(family=family, scale=round(math.exp(rng.uniform(math.log(0.05), 0.0)), 3), poisson=rng.choice([False, True]), drive=drive,
                    steps=_log(rng, 20, 1000 if drive == "run" else 100), read="recording")
    if family == "izhikevich":
        return dict(family=family, neurons=_log(rng, 10000, 1000000), fan=_log(rng, 100, 1000), matrix=rng.choice(["SPARSE", "PROCEDURAL"]),
                    drive=drive, steps=_log(rng, 5, 20), read="recording")
    if family == "plastic":
        return dict(family=family, neurons=_log(rng, 5000, 100000), fan=_log(rng, 100, 500), rule=rng.choice(["STDPTrace", "STDP"]), drive=drive,
                    steps=_log(rng, 20, 100), read="recording")
    if family == "conv":
        return dict(family=family, height=rng.randint(16, 64), width=rng.randint(16, 64), channels_in=rng.randint(1, 16), channels_out=rng.randint(4, 32),
                    kernel=rng.choice([3, 5]), batch=rng.randint(1, 16), steps=rng.randint(20, 50))
    if family == "dense":
        return dict(family=family, inputs=_log(rng, 256, 8192), outputs=_log(rng, 10, 8192), batch=_log(rng, 1, 16), steps=rng.randint(20, 50))
    return dict(family=family, neurons=_log(rng, 10000, 100000), fan=_log(rng, 100, 1000))


# --------------------------------------------------------------------------------------------------------------------
# the networks
# --------------------------------------------------------------------------------------------------------------------
class _Loaded:
    """A loaded model, unloaded with its last reference (a state, or an output that shows its memory)."""

    def __init__(self, model):
        self.model = model

    def __del__(self):
        self.model.unload()


class _DeviceMemory:
    """An Array's device memory for torch.as_tensor()."""

    def __init__(self, loaded, array):
        self.loaded = loaded
        kind = {"float32": "<f4", "uint32": "<i4", "uint8": "|u1"}[array.dtype.name]
        self.__cuda_array_interface__ = dict(shape=(array.count,), typestr=kind, data=(array.ptr, False), version=3)


def _shown(loaded, array):
    return torch.as_tensor(_DeviceMemory(loaded, array), device="cuda")


def _lif_population(model, name, n, v, record, **params):
    pop = model.add_neuron_population(name, n, "LIF", dict(LIF, **params), {"V": v, "RefracTime": 0.0})
    pop.spike_recording_enabled = record
    return pop


def _sparse(model, name, src, trg, weight_update, postsynaptic, snippet, params):
    s = model.add_synapse_population(name, "SPARSE", src, trg, weight_update, postsynaptic, init_sparse_connectivity(snippet, params))
    s.row_stride_multiple = 4
    return s


def _balanced(model, case, record):
    """Excitatory and inhibitory LIF neurons, every pair connected with the same probability; the weights of the 4,000-neuron
    configuration (80 inputs a neuron), scaled with the inputs' number so that larger ones stay balanced."""
    model.dt = 0.1
    n = case["neurons"]
    n_e = n * 4 // 5
    scale = 80.0 / case["fan"]
    pops = {name: _lif_population(model, name, size, init_var("Uniform", {"min": -60.0, "max": -50.0}), record) for name, size in (("E", n_e), ("I", n - n_e))}
    for src, weight, tau in (("E", 0.5, 5.0), ("I", -2.25, 10.0)):
        for trg in "EI":
            _sparse(model, src + trg, pops[src], pops[trg], init_weight_update("StaticPulse", {}, {"g": init_var("Constant", {"constant": weight * scale})}),
                    init_postsynaptic("ExpCurr", {"tau": tau}), "FixedProbability", {"prob": case["fan"] / n})


def _microcircuit_share(case):
    return max(0.1, case["scale"])


def _microcircuit(model, case, record):
    """Eight LIF populations and 54 projections with clipped normal weights and delays; below full size neurons and inputs a neuron are
    reduced alike, and weights and constant input grow to make up for it, as in the configuration."""
    model.dt, model.fuse_postsynaptic_models = 0.1, True
    c = configs
    names = [layer + kind for layer in c.PD_LAYERS for kind in "EI"]
    longest = {k: c.PD_MEAN_DELAY[k] + c.PD_DELAY_SD[k] * c.PD_NORM_Q9999 for k in "EI"}
    slots = int(round(max(longest.values()) / model.dt))
    share = _microcircuit_share(case)
    pops, size = {}, {}
    for name in names:
        size[name] = int(round(case["scale"] * c.PD_NUM[name]))
        full = sum(c.pd_mean_weight(s, name) * c.pd_full_num_inputs(s, name) * c.PD_RATE[s] for s in names) + c.PD_MEAN_W * c.PD_EXT[name] * c.PD_BG_RATE
        pops[name] = _lif_population(model, name, size[name], init_var("Normal", {"mean": -58.0, "sd": 5.0}), record, C=0.25, TauM=10.0, Vrest=-65.0, Vreset=-65.0,
                                     Ioffset=0.001 * 0.5 * (1.0 - math.sqrt(share)) * full, TauRefrac=2.0)
        rate, weight = c.PD_EXT[name] * share * c.PD_BG_RATE, c.PD_MEAN_W / math.sqrt(share)
        if case["poisson"]:
            model.add_current_source(name + "_poisson", "PoissonExp", pops[name], dict(weight=weight, tauSyn=0.5, rate=rate))
        else:
            model.add_current_source(name + "_dc", "DC", pops[name], dict(amp=weight * 0.5 * rate / 1000.0))
    big = float(np.finfo(np.float32).max)
    for trg in names:
        for src in names:
            total = int(round(c.pd_full_num_inputs(src, trg) * share * size[trg]))
            if total <= 0:
                continue
            kind, mean = src[-1], c.pd_mean_weight(src, trg) / math.sqrt(share)
            lo, hi = (0.0, big) if kind == "E" else (-big, 0.0)
            g = init_var("NormalClipped", {"mean": mean, "sd": mean * 0.05 if (src, trg) == ("4E", "23E") else abs(mean * 0.1), "min": lo, "max": hi})
            d = init_var("NormalClippedDelay", {"mean": c.PD_MEAN_DELAY[kind], "sd": c.PD_DELAY_SD[kind], "min": 0.0, "max": longest[kind]})
            s = _sparse(model, src + "_" + trg, pops[src], pops[trg], init_weight_update("StaticPulseDendriticDelay", {}, {"g": g, "d": d}),
                        init_postsynaptic("ExpCurr", {"tau": 0.5}), "FixedNumberTotalWithReplacement", {"num": total})
            s.max_dendritic_delay_timesteps = slots


NOISE_ROWS = 8


def _noise(case, seed):
    n_e = case["neurons"] * 4 // 5
    return {name: netgen.uniform_f32(seed, 12 + k, 0, NOISE_ROWS * size, 5.0, 0.0).reshape(NOISE_ROWS, size)
            for k, (name, size) in enumerate((("E", n_e), ("I", case["neurons"] - n_e)))}


def _izhikevich(model, case, record, noise):
    """Regular-spiking Izhikevich neurons with a fixed number of targets each, 80 % excitatory, driven by an array of noise."""
    matrix, pops = case.get("matrix", "SPARSE"), {}
    for name in "EI":
        pops[name] = model.add_neuron_population(name, noise[name].shape[1], "Izhikevich", IZHIKEVICH, {"V": -65.0, "U": -13.0})
        pops[name].spike_recording_enabled = record
        model.add_current_source(name + "_noise", "ArrayNoise", pops[name]).set_extra_global_param("noise", noise[name])
    scale = 1000.0 / case["fan"]
    for src, lo, hi in (("E", 0.0, 0.5), ("I", -1.0, 0.0)):
        for trg, num in (("E", case["fan"] * 4 // 5), ("I", case["fan"] - case["fan"] * 4 // 5)):
            model.add_synapse_population(src + trg, matrix, pops[src], pops[trg],
                                         init_weight_update("StaticPulse", {}, {"g": init_var("Uniform", {"min": lo * scale, "max": hi * scale})}),
                                         init_postsynaptic("DeltaCurr"), init_sparse_connectivity("FixedNumberPostWithReplacement", {"num": num}))


PLASTIC_STEPS = 100000      # the sources' spike trains are this long: more than anybody steps one state


def _plastic(model, case, record):
    """A balanced network whose excitatory synapses learn; Poisson sources drive it."""
    n = case["neurons"]
    n_e = n * 4 // 5
    size = {"E": n_e, "I": n - n_e}
    pops = {k: _lif_population(model, k, v, init_var("Uniform", {"min": -60.0, "max": -50.0}), record, Ioffset=0.45) for k, v in size.items()}
    n_src, scale = max(10, n // 100), 500.0 / case["fan"]
    rng = np.random.default_rng(model.seed)
    times = np.ceil(np.cumsum(rng.exponential(100.0, (n_src, PLASTIC_STEPS // 100)), axis=1)).astype(np.float32)
    end = np.arange(1, n_src + 1, dtype=np.uint32) * times.shape[1]
    pops["P"] = model.add_neuron_population("P", n_src, "SpikeSourceArray", {}, {"startSpike": end - np.uint32(times.shape[1]), "endSpike": end})
    pops["P"].set_extra_global_param("spikeTimes", times.reshape(-1))
    prob = {"prob": min(1.0, case["fan"] / n_e)}
    g = init_var("Uniform", {"min": 0.0, "max": 0.5 * scale})
    if case["rule"] == "STDP":
        rule = init_weight_update("STDP", dict(STDP_ADDITIVE, Aplus=0.01 * scale, Aminus=0.012 * scale, Wmax=scale), {"g": g})
    else:
        rule = init_weight_update("STDPTrace", dict(STDP_TRACE, aPlus=0.01 * scale, aMinus=0.012 * scale, wMax=scale), {"g": g}, {"preTrace": 0.0}, {"postTrace": 0.0})
    _sparse(model, "EE", pops["E"], pops["E"], rule, init_postsynaptic("ExpCurr", {"tau": 5.0}), "FixedProbability", prob)
    for name, w, tau in (("EI", 0.25, 5.0), ("IE", -1.0, 10.0), ("II", -1.0, 10.0)):
        _sparse(model, name, pops[name[0]], pops[name[1]], init_weight_update("StaticPulse", {}, {"g": init_var("Constant", {"constant": w * scale})}),
                init_postsynaptic("ExpCurr", {"tau": tau}), "FixedProbability", prob)
    _sparse(model, "PE", pops["P"], pops["E"], init_weight_update("StaticPulse", {}, {"g": init_var("Constant", {"constant": 2.0})}),
            init_postsynaptic("ExpCurr", {"tau": 5.0}), "FixedNumberPostWithReplacement", {"num": 100})


def _input_spikes(seed, batch, n, steps, most_hz):
    """Rate-coded samples: every input has a rate of U[0, most_hz) Hz of its own and, per sample, a Poisson train of spikes on a 1 ms
    grid; as a spike source's arrays (start and end of every train, all trains' times, room for the busiest batch)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rate = torch.rand(n, 1, generator=gen, device="cuda") * (most_hz / 1000.0)
    fire = torch.stack([torch.rand(n, steps, generator=gen, device="cuda") < rate for _ in range(batch)]).reshape(batch * n, steps)
    end = torch.cumsum(fire.sum(dim=1), 0)
    times = torch.nonzero(fire)[:, 1].to(torch.float32).cpu().numpy()
    end = end.cpu().numpy().astype(np.uint32)
    start = np.concatenate([np.zeros(1, np.uint32), end[:-1]])
    return start.reshape(batch, n), end.reshape(batch, n), times


def _sources(model, case, n, most_hz):
    start, end, times = _input_spikes(model.seed, case["batch"], n, case["steps"], most_hz)
    pop = model.add_neuron_population("In", n, "SpikeSourceArray", {}, {"startSpike": start, "endSpike": end})
    pop.set_extra_global_param("spikeTimes", times)
    return pop


def _conv(model, case, record):
    h, w, ic, oc, k = (case[q] for q in ("height", "width", "channels_in", "channels_out", "kernel"))
    src = _sources(model, case, h * w * ic, 50.0)
    out = _lif_population(model, "Out", h * w * oc, -60.0, record, Ioffset=0.3)
    shape = dict(conv_kh=k, conv_kw=k, conv_ih=h, conv_iw=w, conv_ic=ic, conv_oh=h, conv_ow=w, conv_oc=oc)
    g = netgen.normal_f32(model.seed, 2, 0, k * k * ic * oc, 0.0, 0.1).reshape(k, k, ic, oc)
    model.add_synapse_population("Layer", "TOEPLITZ", src, out, init_weight_update("StaticPulse", {}, {"g": g}), init_postsynaptic("ExpCurr", {"tau": 5.0}),
                                 init_toeplitz_connectivity("Conv2D", shape))


def _dense(model, case, record):
    src = _sources(model, case, case["inputs"], 100.0)
    out = _lif_population(model, "Out", case["outputs"], -60.0, record, Ioffset=0.3)
    sd = 0.02 * math.sqrt(8192.0 / case["inputs"])
    model.add_synapse_population("Layer", "DENSE", src, out, init_weight_update("StaticPulse", {}, {"g": init_var("Normal", {"mean": 0.0, "sd": sd})}),
                                 init_postsynaptic("ExpCurr", {"tau": 5.0}))


FAMILIES = {"balanced": _balanced, "microcircuit": _microcircuit, "izhikevich": _izhikevich, "plastic": _plastic, "conv": _conv, "dense": _dense,
            "build": _izhikevich}


def _given(case, seed):
    """Arrays that a program has before it describes the model."""
    return (_noise(case, seed),) if case["family"] in ("izhikevich", "build") else ()


def _load(case, seed, given):
    """The case's model, loaded.  A random matrix whose longest row exceeds the space the snippet reserves (one in 10^4) is
    refused by load(); such a model is drawn again."""
    for attempt in range(20):
        model = GeNNModel("float", case["family"], batch_size=case.get("batch", 1), dt=1.0)
        model.seed = int(seed) * 64 + attempt
        record = case["family"] in ("conv", "dense") or "read" in case
        FAMILIES[case["family"]](model, case, record, *given)
        model.build()
        try:
            model.load(num_recording_timesteps=case["steps"] if record else None)
            return _Loaded(model)
        except RuntimeError as e:
            model.unload()
            if "rowStride" not in str(e):
                raise
    raise RuntimeError("no matrix of 20 fits its rows")


class _State:
    pass


def prepare(case, seed):
    """A loaded network as a user's program holds it, and where its state lies in device memory (looked at, never copied)."""
    s = _State()
    s.case, s.seed, s.given, s.loaded = case, seed, _given(case, seed), None
    if case["family"] == "build":
        return s
    s.loaded = _load(case, seed, s.given)
    model = s.model = s.loaded.model
    s.pops = [p for p in model.neuron_populations.values() if p.neuron != "SpikeSourceArray"]
    s.shown = {}
    for p in s.pops:
        for v in ("V", "RefracTime", "U"):
            if v in p.vars:
                s.shown[p.name + "." + v] = _shown(s.loaded, p.vars[v])
        for psm in p.fused_psm:
            s.shown[psm[0].name + ".outPost"] = _shown(s.loaded, psm[0].vars["outPost"])
    if case["family"] == "plastic":
        s.shown["EE.g"] = _shown(s.loaded, model.synapse_populations["EE"].vars["g"])
    if case["family"] in ("conv", "dense"):
        # what a trial starts from, kept on the device
        s.source, s.layer = model.neuron_populations["In"], model.synapse_populations["Layer"]
        out = model.neuron_populations["Out"]
        s.resets = []
        for a in (out.vars["V"], out.vars["RefracTime"], s.layer.vars["outPost"]):
            kept = model._alloc(a.count, np.float32)
            kept.copy_on_device(a)
            s.resets.append((a, kept))
    return s


def _raster(s):
    s.model.pull_recording_buffers_from_device()
    if s.case["read"] == "spikes":
        # spikes of every neuron, and of the population in every step
        out, steps = {}, s.case["steps"]
        for p in s.pops:
            times, ids = p.spike_recording_data[0]
            out[p.name + ".neurons"] = np.bincount(ids, minlength=p.num_neurons)
            out[p.name + ".steps"] = np.bincount(np.rint(times / s.model.dt).astype(np.int64) - (s.model.timestep - steps), minlength=steps)
        return out
    return {p.name + ".recordSpk": p.vars["recordSpk"].view.view(np.int32) for p in s.pops}


def run(s):
    case = s.case
    if case["family"] == "build":
        if s.loaded is not None:
            s.loaded.model.unload()
        s.loaded = _load(case, s.seed, s.given)
        return {name + "." + v: _shown(s.loaded, g.vars[v]) for name, g in s.loaded.model.synapse_populations.items() for v in ("rowLength", "ind", "g")}
    model = s.model
    if case["family"] in ("conv", "dense"):
        # one batch of samples: its input spikes, the layer at rest, the simulation, the output's raster
        for v in ("startSpike", "endSpike", "spikeTimes"):
            s.source.vars[v].push_to_device()
        s.source.vars["spkCnt"].view[:] = 0
        s.source.vars["spkCnt"].push_to_device()
        for a, kept in s.resets:
            a.copy_on_device(kept)
        model.timestep = 0
        model.run(case["steps"])
        model.pull_recording_buffers_from_device()
        return [s.pops[0].vars["recordSpk"].view.view(np.int32), s.shown]
    if case["drive"] == "closed_loop":
        # (the program's answer to a step is made from its spikes; here they are counted)
        counts = [np.zeros(p.num_neurons, np.int32) for p in s.pops]
        for _ in range(case["steps"]):
            model.step_time()
            for count, p in zip(counts, s.pops):
                count[p.current_spikes[0]] += 1
        return [counts, s.shown]
    if case["drive"] == "run":
        model.run(case["steps"])
    else:
        for _ in range(case["steps"]):
            model.step_time()
    return [_raster(s), s.shown]


# --------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct ones may be apart
# --------------------------------------------------------------------------------------------------------------------
def work(case):
    """Synapses: index and weight (and delay) of every synapse of every spiking row, and the written weight of a plastic one.  Neurons:
    the state once in and once out a pass, the noise every step.  The raster as written.  Operations: one add an event and about 15 a
    neuron and step."""
    family, steps = case["family"], case.get("steps", 1)
    if family == "build":
        synapses = case["neurons"] * case["fan"]
        return {"bytes": 8.0 * synapses, "flops": 10.0 * synapses}
    if family == "conv":
        n_in = case["height"] * case["width"] * case["channels_in"] * case["batch"]
        n = case["height"] * case["width"] * case["channels_out"] * case["batch"]
        spikes = n_in * 0.025 * steps
        taps = case["kernel"] ** 2 * case["channels_out"]
        return {"bytes": 12.0 * n_in + 4.0 * spikes + n * 24.0 + n / 8.0 * steps + 4.0 * taps * case["channels_in"], "flops": spikes * taps + 15.0 * n * steps}
    if family == "dense":
        spikes = case["inputs"] * 0.05 * steps * case["batch"]
        n = case["outputs"] * case["batch"]
        events = spikes * case["outputs"]
        return {"bytes": 4.0 * min(case["inputs"] * case["outputs"] * steps, events) + 12.0 * case["inputs"] * case["batch"] + 4.0 * spikes + n * 24.0 + n / 8.0 * steps,
                "flops": events + 15.0 * n * steps}
    # spikes a neuron and step, as these networks run
    if family == "microcircuit":
        n, fan, rate, per_event = 77169 * case["scale"], 3870 * _microcircuit_share(case), 3.2e-4, 9.0
    elif family == "balanced":
        n, fan, rate, per_event = case["neurons"], case["fan"], 1.3e-3, 8.0
    elif family == "izhikevich":
        n, fan, rate, per_event = case["neurons"], case["fan"], 1.3e-2, 8.0 if case["matrix"] == "SPARSE" else 0.0
    else:
        n, fan, rate, per_event = case["neurons"], case["fan"] * 1.25, 1.0e-2, 12.0
    events = n * fan * rate * steps
    noise = 4.0 * n * steps if family == "izhikevich" else 0.0
    return {"bytes": events * per_event + n * 24.0 + noise + n / 8.0 * steps, "flops": events + 15.0 * n * steps}


def tolerance(case):
    """Matrices are whole numbers and single roundings.  Elsewhere inputs are fp32 sums in any order: 1e-5, and spikes are the same but
    for a neuron that such a sum puts on the other side of its threshold."""
    if case["family"] == "build":
        return {"rel": 1e-6, "differ": 0.0}
    return {"rel": 1e-5, "max": 1e-3, "differ": 1e-4}
