"""Workloads of the cerebellar-scaffold engine, as programs that use it run them.

Every case drives one network (or a batch of networks) through the Python binding:
describe, initialize, then passes of the simulation that carry on from each other.
The networks are the seeded scaffold generator's, of the sizes the tests and the
benchmark use (9.9k cells, 0.25x to 16x of the 96.7k-cell scaffold); a pass is

  step    one exchange step (1 ms) of a controller that closes its loop every
          millisecond: new input rates, loop_n_steps(1), the step's spike counts
  window  one iteration of the reference's driver loop: input rates, loop_n_steps
          over a hand-off window of 25 steps with the output train, running totals
  raster  a window, then the list of fired neurons of each of its steps
  trial   several windows of the driver loop, then the whole neuron state
  run     a stretch of steps in one call without hand-offs, then the neuron state
  learn   a trial of a network with a plasticity rule, then its multipliers too
  batch   several networks of uneven size advanced together by one Batch, then the
          state and totals of each

Connectivity is fixed for a size, as a program loads one connectome; the seed draws
the synaptic multipliers, the initial potentials, the stimulus streams and, where
they change from window to window, the input rates.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import __graft_entry__  # noqa: E402

T_PRINT, WINDOW = 50, 25          # the reference's main.cu
FULL = 96737                      # cells of the 1x scaffold
SMALL_COUNTS = (8800, 700, 7, 22, 60, 60, 2, 240)  # the 9.9k-cell test network


def _pkg():
    pkg = __graft_entry__.load_package()
    pkg.load_library()
    return pkg


# ------------------------------------------------------------------ the cases
def _case(name, kind, **more):
    """scale: area relative to the 96.7k-cell scaffold (0: the 9.9k-cell test network);
    dense: 1 the reference connectome's fan-ins, 0 the rule-text density; weights:
    storage of the multipliers (unit: none, every synapse 1, as the reference's .dat
    loader gives); bits: column index width; rate: mossy background in Hz (0: drawn
    by the seed, another for each window); steps: exchange steps of a pass."""
    c = {"name": name, "kind": kind, "scale": 1.0, "dense": 1, "weights": "f32", "bits": 32, "rate": 4.0,
         "steps": WINDOW, "rule": ""}
    c.update(more)
    return c


def listed():
    return [
        # smallest call: a controller exchanging with the test-size network every 1 ms
        _case("step_10k", "step", scale=0.0, rate=0.0, steps=1),
        # the driver loop on the test-size network, the controller changing the input
        _case("window_10k", "window", scale=0.0, rate=0.0),
        # the driver loop on the reference-size scaffold: the benchmark's headline
        _case("window_97k", "window"),
        # the same with the rasters collected, neuron lists per step
        _case("raster_97k", "raster"),
        # a quarter second of the reference's own description (unit multipliers)
        _case("trial_97k_unit", "trial", weights="unit", steps=250),
        # the rule-text density in the compact forms a memory-bound user picks
        _case("trial_97k_bf16_idx16", "trial", dense=0, weights="bf16", bits=16, steps=250),
        # strong mossy drive: an order of magnitude more spikes
        _case("trial_97k_60hz", "trial", rate=60.0, steps=250),
        # the reference's parallel-fibre-to-Purkinje rule, the benchmark's plastic leg
        _case("learn_97k_teacher", "learn", rule="teacher", steps=250),
        # four plastic terms on lane-gathered synapses of a quarter-size network
        _case("learn_24k_hebb", "learn", scale=0.25, rule="hebb", steps=100),
        # a parameter sweep: uneven instances, mossy rates 1-60 Hz
        _case("batch_8_bf16", "batch", weights="bf16", rate=0.0, steps=200),
        # networks beyond the caches, advanced without hand-offs
        _case("run_4x_f32", "run", scale=4.0, steps=100),
        _case("run_16x_fp8_idx16", "run", scale=16.0, weights="fp8", bits=16, steps=100),
    ]


def draw(rng):
    def log_uniform(a, b):
        return math.exp(rng.uniform(math.log(a), math.log(b)))

    kind = rng.choice(["step", "window", "window", "raster", "trial", "trial", "run", "learn", "batch"])
    top = {"step": 2.0, "window": 4.0, "raster": 2.0, "trial": 3.0, "run": 4.0, "learn": 1.2, "batch": 1.5}[kind]
    steps = {"step": 1, "window": WINDOW, "raster": WINDOW, "trial": WINDOW * rng.randint(2, 10),
             "run": rng.randint(5, 120), "learn": WINDOW * rng.randint(1, 6), "batch": rng.randint(20, 160)}[kind]
    weights = rng.choice(["f32", "f32", "bf16", "fp8", "unit"])
    return {"kind": kind, "scale": round(log_uniform(0.06, top), 3), "dense": rng.choice([0, 1, 1]),
            "weights": "f32" if kind == "learn" else weights, "bits": rng.choice([32, 32, 16]),
            "rate": 0.0 if kind == "batch" else rng.choice([0.0, round(log_uniform(1.0, 60.0), 2)]),
            "steps": steps, "rule": rng.choice(["teacher", "template", "hebb"]) if kind == "learn" else ""}


def _instances(case):
    """Scales of the networks of a case."""
    if case["kind"] != "batch":
        return [case["scale"]]
    return [round(s * case["scale"], 3) for s in (0.25, 0.25, 0.25, 0.5, 0.5, 1.0, 1.0, 2.0)]


# ------------------------------------------------------------------- networks
_GRAPHS = {}


def _graph(scale, dense):
    """The network description of one size: populations, CSR projections in index
    order, stimuli.  Described once by the generator; programs keep it."""
    key = (scale, dense)
    if key not in _GRAPHS:
        if len(_GRAPHS) > 24:
            _GRAPHS.clear()
        pkg = _pkg()
        cfg = pkg.synth_preset(1 if scale > 0 else 0)
        cfg.weight_jitter = 0
        if scale > 0:
            cfg.scale = scale
            cfg.connectome = dense
            cfg.burst_n_mf = max(1, int(round(50 * scale)))
        else:
            for i, n in enumerate(SMALL_COUNTS):
                cfg.counts[i] = n
        env = pkg.NetworkEnvironment(1, 7, 16, 2)
        env.describe_synthetic(cfg)
        info = env.info()
        pops, projs, stims = [], [], []
        for i in range(info.n_populations):
            p = env.population(i)
            pops.append({"type": p.type, "name": p.name.decode(), "num": p.num, "kind": p.device_type,
                         "par": (p.Cm, p.El, p.dt_ref, p.Ie, p.Vr, p.Vth, p.gL),
                         "ch": [x for c in range(p.c_num) for x in (p.w[c], p.E[c], p.g_bar[c], p.tau[c])]})
        for i in range(info.n_projections):
            p = env.projection(i)
            if p.pre < 0:
                continue
            row_ptr, col, _ = env.projection_csr(i)
            projs.append({"index": i, "type": p.type, "pre": p.pre, "post": p.post, "w": p.initial_weight,
                          "delay": p.delay, "row_ptr": row_ptr, "col": np.ascontiguousarray(col)})
        for i in range(info.n_stimuli):
            s, fan, ids = env.stimulus(i)
            stims.append({"pop": s.pop, "fan": fan, "ids": np.ascontiguousarray(ids), "burst_hz": s.func.burst_hz,
                          "on": s.func.burst_on, "off": s.func.burst_off})
        env.finalize()
        _GRAPHS[key] = {"pops": pops, "projs": projs, "stims": stims}
    return _GRAPHS[key]


def _multipliers(graph, case, seed):
    """Per projection the multipliers U(0.8, 1.2) of this seed (None: unit).  The
    target of a Hebb rule, whose multipliers the rule keeps in [0, 1], has U(0.4, 0.6)."""
    if case["weights"] == "unit":
        return [None] * len(graph["projs"])
    gen = torch.Generator().manual_seed(seed)
    out = []
    for p in graph["projs"]:
        v = torch.rand(len(p["col"]), generator=gen, dtype=torch.float32)
        if case["rule"] == "hebb" and p["type"] == 15:
            v.mul_(0.2).add_(0.4)
        else:
            v.mul_(0.4).add_(0.8)
        out.append(v.numpy())
    return out


def _rates(case, seed, instance=0):
    """Mossy rates (Hz) of successive windows; one value where the rate is fixed."""
    if case["rate"] > 0:
        return [case["rate"]]
    gen = torch.Generator().manual_seed(1000 * seed + instance)
    n = 1 if case["kind"] == "batch" else 16
    top = 60.0 if case["kind"] == "batch" else 12.0
    return [float(x) for x in torch.exp(torch.rand(n, generator=gen, dtype=torch.float64) * math.log(top))]


def _rule(pkg, case):
    """(rule, target type, teacher type, coefficients {slot: (c, a, b)}, window): the
    reference's shipped rule, its code-generation template's, and a four-term Hebb rule."""
    if case["rule"] == "teacher":
        return pkg.STDP_TEACHER, 0, 11, {pkg.A1_J: (0.0, 0.0, 0.0), pkg.A2_JI: (-0.01, 0.0, 0.0)}, 50
    if case["rule"] == "template":
        return pkg.STDP_TEACHER, 0, 11, {pkg.A1_J: (0.0, 0.001, 1.0), pkg.A2_JI: (0.0, 0.01, 0.0)}, 50
    if case["rule"] == "hebb":
        return pkg.STDP_HEBB, 15, -1, {pkg.A0: (0.0001, 0.0, 0.0), pkg.A1_I: (-0.002, 0.0, 0.0),
                                       pkg.A1_J: (0.0, 0.004, 0.5), pkg.A2_JI: (0.001, 0.0, 0.0)}, 20
    return None


def _seeds(seed, instance):
    return 2 * (1000 * seed + instance) + 1, 5_000_000_000 + 16 * (1000 * seed + instance)  # neurons, stimuli


def _build(pkg, case, scale, seed, instance):
    graph = _graph(scale, case["dense"])
    rule = _rule(pkg, case)
    env = pkg.NetworkEnvironment(1, len(graph["pops"]), 16, max(1, len(graph["stims"])), 1 if rule else 0)
    order = [i for i, p in enumerate(graph["pops"]) if p["kind"] == pkg.NORMAL]
    order += [i for i in reversed(range(len(graph["pops"]))) if graph["pops"][i]["kind"] != pkg.NORMAL]
    for i in order:  # NORMAL populations are indexed from the front, the others from the back
        p = graph["pops"][i]
        env.set_neuron_params(p["type"], p["name"], 0, p["num"], *p["par"], p["kind"], p["ch"])
    values = _multipliers(graph, case, 1000 * seed + instance)
    out = [k for k, p in enumerate(graph["projs"]) if graph["pops"][p["post"]]["kind"] == pkg.OUTPUT]
    index = {}
    for k in [k for k in range(len(graph["projs"])) if k not in out] + out[::-1]:
        p = graph["projs"][k]
        index[p["type"]] = env.set_connectivity_csr(p["type"], graph["pops"][p["pre"]]["num"],
                                                    graph["pops"][p["post"]]["num"], p["pre"], p["post"], p["w"],
                                                    float(p["delay"]), p["row_ptr"], p["col"], values[k])
    neuron_seed, stim_seed = _seeds(seed, instance)
    rate = _rates(case, seed, instance)[0]
    for i, s in enumerate(graph["stims"]):
        f = pkg.StimFunc()
        f.poisson_hz, f.poisson_on, f.poisson_off = rate, 0.0, math.inf
        f.poisson_hz_from_freq = 1
        if i > 0:
            f.burst_hz, f.burst_on, f.burst_off = s["burst_hz"], s["on"], s["off"]
        f.seed = stim_seed + i
        env.set_input_stim_ids(s["pop"], s["ids"], f, s["fan"])
    if rule:
        kind, target, teacher, coef, window = rule
        env.set_plasticity_affine(kind, index[target], index.get(teacher, -1), coef, window)
    env.set_option("neuron_seed", neuron_seed)
    env.set_option("weight_precision", {"bf16": pkg.WEIGHTS_BF16, "fp8": pkg.WEIGHTS_FP8}.get(case["weights"],
                                                                                              pkg.WEIGHTS_F32))
    env.set_option("index_bits", case["bits"])
    env.initialize(T_PRINT, 1 if case["kind"] == "step" else WINDOW)
    return env, index


def prepare(case, seed):
    pkg = _pkg()
    envs, index = [], {}
    for i, scale in enumerate(_instances(case)):
        env, index = _build(pkg, case, scale, seed, i)
        envs.append(env)
    rates = _rates(case, seed)
    info = envs[0].info()
    state = {"kind": case["kind"], "steps": case["steps"], "envs": envs, "t": 0, "calls": 0,
             "cells": info.total_neurons, "freqs": [[r] * info.n_stimuli for r in rates], "batch": None,
             "plastic": -1}
    if case["rule"]:
        state["plastic"] = index[_rule(pkg, case)[1]]
    if case["kind"] == "batch":
        state["batch"] = pkg.Batch(envs)
    return _State(state)


class _State(dict):
    """The state of a case; a program that ends lets its batch go before its networks."""

    def __del__(self):
        try:
            if self["batch"] is not None:
                self["batch"].destroy()
            for env in self["envs"]:
                env.finalize()
        except Exception:
            pass


# ------------------------------------------------------------------ one pass
def _window(state, n):
    """Input rates of the next window, its n steps, the output train."""
    env = state["envs"][0]
    env.set_input_freq(state["freqs"][state["calls"] % len(state["freqs"])])
    train = env.loop_n_steps(state["t"], n)
    state["t"] += n
    state["calls"] += 1
    return train


def _whole(env):
    V, g, refr = env.state()
    spikes, events = env.totals()
    return {"V": V, "g": g, "refr": refr, "spikes": spikes.astype(np.int64), "events": int(events)}


def run(state):
    kind, steps, env = state["kind"], state["steps"], state["envs"][0]
    if kind == "step":
        train = _window(state, 1)
        counts, events = env.counts(state["t"] - 1)
        return {"train": train, "counts": counts, "events": int(events)}
    if kind == "window":
        train = _window(state, steps)
        spikes, events = env.totals()
        return {"train": train, "spikes": spikes.astype(np.int64), "events": int(events)}
    if kind == "raster":
        train = _window(state, steps)
        cap = max(64, state["cells"] // 16)
        ids, n = np.full((steps, cap), -1, np.int32), np.zeros(steps, np.int32)
        for i in range(steps):
            step_ids, n[i] = env.fired(state["t"] - steps + i, cap)
            ids[i, :len(step_ids)] = step_ids
        return {"train": train, "fired": ids, "n": n}
    if kind == "batch":
        state["batch"].run(steps)
        return [_whole(e) for e in state["envs"]]
    if kind == "run":
        env.loop_n_steps(state["t"], steps, want_output=False)
        state["t"] += steps
        return _whole(env)
    trains = [_window(state, WINDOW) for _ in range(steps // WINDOW)]
    out = {"trains": np.stack(trains), **_whole(env)}
    if kind == "learn":
        out["multipliers"] = env.projection_csr(state["plastic"])[2]
    return out


# --------------------------------------------------------------- work of a pass
def work(case):
    """Per step every neuron's 16-byte state read and written and its spike bit; the
    synapses once per pass, as a cache may keep them.  Ten Euler sub-steps of about
    20 operations per neuron and step, a sum per synapse and step."""
    wb = {"unit": 0, "f32": 4, "bf16": 2, "fp8": 1}[case["weights"]]
    total = {"bytes": 0.0, "flops": 0.0}
    for scale in _instances(case):
        cells = FULL * scale if scale > 0 else 9900
        fan_in = (43.7 if case["dense"] else 31.4) if scale > 0 else 20.5
        synapses = cells * fan_in
        total["bytes"] += case["steps"] * cells * (32 + 1 / 8) + synapses * (case["bits"] / 8 + wb) + cells * 16
        total["flops"] += case["steps"] * (cells * 200 + synapses)
    return total


# ----------------------------------------------- the same simulation in 64 bits
def _philox(seed, stream, block):
    """Philox4x32-10 (Salmon et al., SC'11): the four words of `block` of each stream."""
    u = np.uint64
    low = u(0xFFFFFFFF)
    c = [np.full(stream.shape, block & 0xFFFFFFFF, u), np.full(stream.shape, block >> 32, u), stream.astype(u),
         np.zeros(stream.shape, u)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        p0, p1 = c[0] * u(0xD2511F53), c[2] * u(0xCD9E8D57)
        c = [(p1 >> u(32)) ^ c[1] ^ u(k0), p1 & low, (p0 >> u(32)) ^ c[3] ^ u(k1), p0 & low]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _uniform(words):
    inv = np.float32(2.3283064365386963e-10)
    return (inv + words.astype(np.float32) * inv).astype(np.float64)


def _stored(values, weights):
    """Multipliers as the storage holds them, in float64, with the factor of a row sum."""
    if values is None or weights not in ("bf16", "fp8"):
        return values, 1.0
    v = torch.from_numpy(values)
    if weights == "bf16":
        q = v.to(torch.bfloat16).double()
    else:
        scale = 2.0 ** math.ceil(math.log2(float(v.abs().max()) / 448.0))
        q = (v / scale).to(torch.float8_e4m3fn).double() * scale
    return q.numpy(), float(np.float32(values.astype(np.float64).sum() / float(q.sum())))


class _Sim:
    """The scaffold's exchange step in float64 with plain tensor operations."""

    def __init__(self, case, scale, seed, instance):
        graph = _graph(scale, case["dense"])
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.graph, self.n, self.history = graph, 0, []
        nums = [p["num"] for p in graph["pops"]]
        self.base = np.concatenate([[0], np.cumsum(nums)])
        total = int(self.base[-1])
        pop = np.repeat(np.arange(len(nums)), nums)

        def per_neuron(f):
            return torch.tensor([float(f(p)) for p in graph["pops"]], dtype=torch.float64)[pop].to(self.dev)

        f32 = np.float32
        par = ["Cm", "El", "dt_ref", "Ie", "Vr", "Vth", "gL"]
        P = {k: per_neuron(lambda p, i=i: f32(p["par"][i])) for i, k in enumerate(par)}
        P["dtc"] = torch.where(P["Cm"] > 0, 0.1 / P["Cm"], torch.zeros_like(P["Cm"]))
        self.P = P
        self.ref_step = per_neuron(lambda p: int(float(f32(p["par"][2])) / 0.1)).to(torch.int32)
        self.ch = [{"E": per_neuron(lambda p: p["ch"][4 * c + 1] if p["ch"] else 0),
                    "gw": per_neuron(lambda p: f32(p["ch"][4 * c + 2]) * f32(p["ch"][4 * c]) if p["ch"] else 0),
                    "dtt": per_neuron(lambda p: 0.1 / float(f32(p["ch"][4 * c + 3])) if p["ch"] else 0)}
                   for c in range(2)]
        for c in self.ch:
            c["exc"] = c["E"] > P["El"]
        self.active = per_neuron(lambda p: 1 if p["ch"] else 0).bool()
        self.neuron_seed, self.stim_seed = _seeds(seed, instance)
        # the second uniform number of each neuron's stream starts the first trial
        U = torch.from_numpy(_uniform(_philox(self.neuron_seed, np.arange(total, dtype=np.uint64), 0)[1])).to(self.dev)
        self.V = P["Vr"] + (P["Vth"] - P["Vr"]) * U
        self.g = [torch.zeros(total, dtype=torch.float64, device=self.dev) for _ in range(2)]
        self.refr = torch.zeros(total, dtype=torch.int32, device=self.dev)
        values = _multipliers(graph, case, 1000 * seed + instance)
        self.projs = []
        for p, v in zip(graph["projs"], values):
            stored, factor = _stored(v, "f32" if case["rule"] else case["weights"])
            post = np.repeat(np.arange(len(p["row_ptr"]) - 1), np.diff(p["row_ptr"])) + self.base[p["post"]]
            pre = p["col"].astype(np.int64) + self.base[p["pre"]]
            w = np.ones(len(pre)) if stored is None else stored.astype(np.float64)
            self.projs.append({"pre": torch.from_numpy(pre).to(self.dev), "post": torch.from_numpy(post).to(self.dev),
                               "w": torch.from_numpy(w).to(self.dev), "W": abs(float(f32(p["w"]))) * factor,
                               "exc": p["w"] > 0, "delay": p["delay"], "type": p["type"], "def": p})
        self.rule = _rule(_pkg(), case)

    def spikes_at(self, step):
        return self.history[step] if 0 <= step < len(self.history) else None

    def stimulus(self, out, rate):
        n = self.n
        for i, s in enumerate(self.graph["stims"]):
            entries = np.arange(len(s["fan"]) - 1, dtype=np.uint64)
            words = [w for b in range(3) for w in _philox(self.stim_seed + i, entries, 3 * n + b)]
            fires = np.zeros(len(entries), bool)
            for k in range(10):
                t, r = float(np.float32(n + k * 0.1)), _uniform(words[k])
                fires |= r < float(np.float32(rate)) / 1000.0 * 0.1
                if i > 0 and s["on"] <= t < s["off"]:
                    fires |= r < float(np.float32(s["burst_hz"])) / 1000.0 * 0.1
            ids = torch.from_numpy(s["ids"].astype(np.int64) + self.base[s["pop"]]).to(self.dev)
            out[ids] = torch.from_numpy(np.repeat(fires, np.diff(s["fan"]))).to(self.dev)

    def step(self, rate):
        fired = torch.zeros(self.V.shape, dtype=torch.bool, device=self.dev)
        self.stimulus(fired, rate)
        dg = [torch.zeros_like(self.V), torch.zeros_like(self.V)]
        for p in self.projs:
            spikes = self.spikes_at(self.n - p["delay"])
            if spikes is not None:
                on = spikes[p["pre"]]
                dg[0 if p["exc"] else 1].index_add_(0, p["post"], torch.where(on, p["w"] * p["W"], 0.0))
        P, spk = self.P, torch.zeros_like(fired)
        for k in range(10):
            current = sum(g * (self.V - c["E"]) for g, c in zip(self.g, self.ch))
            du = P["dtc"] * (P["Ie"] - P["gL"] * (self.V - P["El"]) - current)
            for j, c in enumerate(self.ch):
                add = c["gw"] * torch.where(c["exc"], dg[0], dg[1]) if k == 0 else 0.0
                self.g[j] = self.g[j] - c["dtt"] * self.g[j] + add
            over = (self.V > P["Vth"]) & self.active
            spk |= over
            self.refr = torch.where(over, self.ref_step, (self.refr - 1).clamp(min=0))
            self.V = torch.where(self.active, torch.where(self.refr > 0, P["Vr"], self.V + du), self.V)
        self.history.append(torch.where(self.active, spk, fired))
        if self.rule:
            self.learn()
        self.n += 1

    def learn(self):
        kind, target, teacher, coef, window = self.rule
        by_type = {p["type"]: p for p in self.projs}
        p, n = by_type[target], self.n
        post_base = int(self.base[p["def"]["post"]])
        if kind == _pkg().STDP_HEBB:
            trigger = self.history[n][p["post"]]
        else:
            t = by_type[teacher]
            start, end = t["def"]["row_ptr"][:-1], t["def"]["row_ptr"][1:]
            first = np.where(end > start, t["def"]["col"][np.minimum(start, len(t["def"]["col"]) - 1)], 0)
            spikes = self.spikes_at(n - t["delay"])
            if spikes is None:
                spikes = torch.zeros_like(self.history[0])
            row = spikes[torch.from_numpy(first.astype(np.int64) + self.base[t["def"]["pre"]]).to(self.dev)]
            row = row & torch.from_numpy(end > start).to(self.dev)
            trigger = row[p["post"] - post_base]
        past = [self.spikes_at(n - p["delay"] - s) for s in range(window)]
        count = sum(x.to(torch.float64) for x in past if x is not None) if past[0] is not None else None
        w = p["w"]
        value = {slot: c + a * (b - w) for slot, (c, a, b) in coef.items()}
        dw = torch.zeros_like(w)
        if 0 in value:
            dw += value[0]
        if 2 in value and past[0] is not None:
            dw += torch.where(past[0][p["pre"]], value[2], 0.0)
        if 1 in value:
            dw += torch.where(trigger, value[1], 0.0)
        if 3 in value and count is not None:
            dw += torch.where(trigger, value[3] * count[p["pre"]], 0.0)
        p["w"] = (w + dw).clamp(0.0, 1.0) if kind == _pkg().STDP_HEBB else (w + dw).clamp(min=0.0)


def exact(case, seed):
    """Potentials, conductances and multipliers after the pass.  Spikes, counters and
    trains are whole numbers.  Above 16 Hz of mossy drive the granule layer's Euler
    rule leaves its stable range (DT g / Cm > 2) and has no value to converge to; the
    largest network takes too long."""
    if case["kind"] in ("step", "window", "raster"):
        return None
    if max(_instances(case)) > 8:
        return None
    outs = []
    for i, scale in enumerate(_instances(case)):
        rates = _rates(case, seed, i)
        if max(rates) > 16.0:
            outs.append(None)
            continue
        sim = _Sim(case, scale, seed, i)
        for n in range(case["steps"]):
            sim.step(rates[(n // WINDOW) % len(rates)] if case["kind"] in ("trial", "learn") else rates[0])
        out = {"trains": None, "V": sim.V.cpu().numpy(),
               "g": torch.stack(sim.g, 1).reshape(-1).cpu().numpy(), "refr": None, "spikes": None, "events": None}
        if case["kind"] != "trial" and case["kind"] != "learn":
            del out["trains"]
        if case["kind"] == "learn":
            target = _rule(_pkg(), case)[1]
            out["multipliers"] = next(p["w"] for p in sim.projs if p["type"] == target).cpu().numpy()
        outs.append(out)
    if all(o is None for o in outs):
        return None
    return outs if case["kind"] == "batch" else outs[0]
