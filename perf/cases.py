"""Cases of the framework's main path, timed as a user's program runs it:
networks built with Create/Connect, advanced with Simulate and read back,
through the Python module and the C library behind it.

Sizes are those of the repository's own configurations and tests
(neurongpu_amd/workloads.py, bench.py, tests/netbuild.py) and the range
between them.  Weights are multiples of 1/256 nS (or whole pA), so that the
synaptic sums are exact in any order and a recurrent network has one spike
train whatever the order of its float additions; the plastic network is the
exception (its weights are products of exponentials).

The library holds one network per loaded library, so every state that is
alive has a copy of the library of its own (the first one has the in-tree
file itself).
"""
import ctypes
import importlib.util
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from neurongpu_amd import neurongpu as _first
from neurongpu_amd import workloads as wl

DT = 0.1                      # ms, the framework's default time step
W = 1.0 / 256.0               # unit of the conductance weights (nS)


def listed():
    return [
        # a whole small script: build, record two variables of ten neurons,
        # simulate, read the rows (latency, launches, set-up)
        {"name": "script_1k", "kind": "script", "n": 1000, "k": 100,
         "rate": 8000.0, "ms": 20.0},
        # the smallest configuration (1000 AdEx neurons, in-degree 100, one
        # Poisson generator a neuron), advanced 10 ms at a time
        {"name": "adex_1k", "kind": "adex", "active": False, "n": 1000,
         "k": 100, "rate": 8000.0, "gens": "own", "tol": 1e-3, "ms": 10.0,
         "settle": 0.0},
        # the network-statistics test at 10000 neurons, spiking
        {"name": "adex_10k_active", "kind": "adex", "active": True,
         "n": 10000, "k": 1000, "rate": 20000.0, "gens": "one", "tol": 1e-6,
         "ms": 10.0, "settle": 100.0},
        # the headline configuration: 1e6 neurons, 1e9 synapses, silent
        {"name": "adex_1m", "kind": "adex", "active": False, "n": 1000000,
         "k": 1000, "rate": 8000.0, "gens": "one", "tol": 1e-3, "ms": 200.0,
         "settle": 0.0},
        # the same size under the stronger drive of the benchmark network
        # (about 30 spikes/s a neuron)
        {"name": "adex_1m_active", "kind": "adex", "active": True,
         "n": 1000000, "k": 1000, "rate": 20000.0, "gens": "one",
         "tol": 1e-6, "ms": 100.0, "settle": 100.0},
        # three receptor ports, current-based synapses, 8 models more run
        # through the same one-launch RK5 kernels
        {"name": "psc_20k", "kind": "psc", "model": "aeif_psc_exp",
         "n": 20001, "k": 200, "ports": 2, "rate": 8000.0, "ms": 20.0,
         "settle": 20.0},
        # the layered column of current-based neurons at a tenth of its size
        {"name": "iaf_8k", "kind": "iaf", "scale": 0.1, "ms": 20.0,
         "settle": 50.0},
        # and at full size (77169 neurons, about 6e8 synapses)
        {"name": "iaf_77k", "kind": "iaf", "scale": 1.0, "ms": 50.0,
         "settle": 50.0},
        # plasticity: 2e5 AdEx neurons, STDP on the E -> E synapses
        {"name": "stdp_200k", "kind": "stdp", "n": 200000, "k": 500,
         "rate": 8000.0, "ms": 50.0, "settle": 60.0},
        # 64 independent networks in one group
        {"name": "ensemble_64", "kind": "ensemble", "inst": 64,
         "n_lo": 5000, "n_hi": 50000, "ms": 50.0},
        # network construction alone: rules, delays, sorted synapse store
        {"name": "build_200k", "kind": "build", "n": 200000, "k": 500},
        # the step-size proposer's training: minibatches of logged samples
        {"name": "proposer_train", "kind": "train", "n": 1000000,
         "batch": 8192, "iters": 50},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["script", "adex", "adex", "active", "psc", "iaf",
                       "stdp", "ensemble", "build", "train"])
    if kind == "script":
        return {"kind": kind, "n": int(_log(rng, 100, 4000)),
                "k": rng.randint(10, 80), "rate": rng.uniform(4e3, 1e4),
                "ms": float(rng.randint(5, 20))}
    if kind == "adex":
        n = int(_log(rng, 300, 900000))
        return {"kind": "adex", "active": False, "n": n,
                "k": 5 * int(_log(rng, 20, min(1000, n // 5)) / 5),
                "rate": rng.uniform(4e3, 8e3),
                "gens": rng.choice(["one", "own"]) if n <= 50000 else "one",
                "tol": 1e-3, "ms": float(rng.randint(5, 40)), "settle": 0.0}
    if kind == "active":
        n = int(_log(rng, 2000, 600000))
        return {"kind": "adex", "active": True, "n": n,
                "k": 5 * rng.randint(40, min(200, n // 25)),
                "rate": 20000.0, "gens": "one",
                "tol": rng.choice([1e-3, 1e-6]),
                "ms": float(rng.randint(5, 20)), "settle": 30.0}
    if kind == "psc":
        return {"kind": kind,
                "model": rng.choice(["aeif_psc_exp", "aeif_psc_alpha",
                                     "aeif_cond_alpha"]),
                "n": int(_log(rng, 500, 100000)), "k": rng.randint(20, 80),
                "ports": rng.randint(2, 4), "rate": 8000.0,
                "ms": float(rng.randint(5, 20)), "settle": 5.0}
    if kind == "iaf":
        return {"kind": kind, "scale": _log(rng, 0.02, 0.7),
                "ms": float(rng.randint(5, 25)), "settle": 30.0}
    if kind == "stdp":
        return {"kind": kind, "n": 5 * int(_log(rng, 1000, 30000)),
                "k": 5 * rng.randint(10, 80), "rate": 8000.0,
                "ms": float(rng.randint(5, 15)), "settle": 60.0}
    if kind == "ensemble":
        lo = int(_log(rng, 500, 8000))
        return {"kind": kind, "inst": rng.randint(2, 32), "n_lo": lo,
                "n_hi": 4 * lo, "ms": float(rng.randint(5, 30))}
    if kind == "build":
        n = int(_log(rng, 2000, 150000))
        return {"kind": kind, "n": n, "k": rng.randint(20, 400)}
    n = int(_log(rng, 5000, 600000))
    return {"kind": "train", "n": n, "batch": int(_log(rng, 300, 8192)),
            "iters": rng.randint(5, 50)}


# ---------------------------------------------------------------------
# one loaded library per live state
# ---------------------------------------------------------------------
_free, _dir = [], []


def _bind(ng):
    """The library's bulk reads, through its C interface."""
    lib = ctypes.CDLL(ng.lib_path)
    lib.NeuronGPU_GetNeuronVar.restype = ctypes.POINTER(ctypes.c_float)
    lib.NeuronGPU_GetNeuronVar.argtypes = [ctypes.c_int, ctypes.c_int,
                                           ctypes.c_char_p]
    lib.NeuronGPU_GetNeuronIntVar.restype = ctypes.POINTER(ctypes.c_int)
    lib.NeuronGPU_GetNeuronIntVar.argtypes = [ctypes.c_int, ctypes.c_int,
                                              ctypes.c_char_p]
    ng.SetVerbosityLevel(0)
    return ng, lib


def _library():
    if _free:
        return _free.pop()
    if not _dir:
        _dir.append(None)
        return _bind(_first)
    if _dir[0] is None:
        _dir[0] = tempfile.mkdtemp(prefix="neurongpu_")
    path = os.path.join(_dir[0], "libneurongpu_%d.so" % len(_dir))
    _dir.append(path)
    shutil.copyfile(_first.lib_path, path)
    spec = importlib.util.spec_from_file_location(
        "neurongpu_copy_%d" % len(_dir), _first.__file__)
    ng = importlib.util.module_from_spec(spec)
    before = os.environ.get("NEURONGPU_LIB")
    os.environ["NEURONGPU_LIB"] = path
    try:
        spec.loader.exec_module(ng)
        got = _bind(ng)
    finally:
        if before is None:
            del os.environ["NEURONGPU_LIB"]
        else:
            os.environ["NEURONGPU_LIB"] = before
        os.unlink(path)
    return got


class State:
    """A network (or the proposer) in a library of its own."""

    def __init__(self, case):
        self.case = case
        self.ng, self.lib = _library()
        self.neuron = None

    def variables(self):
        """Every state variable of the neurons, by name."""
        i0, n, out = self.neuron.i0, self.neuron.n, {}
        for name in self.names:
            p = self.lib.NeuronGPU_GetNeuronVar(i0, n, name.encode())
            if not p:
                raise RuntimeError(self.ng.GetErrorMessage())
            out[name] = np.ctypeslib.as_array(
                p, (n, self.ng.GetNeuronVarSize(i0, name)))
        return out

    def counts(self):
        p = self.lib.NeuronGPU_GetNeuronIntVar(self.neuron.i0, self.neuron.n,
                                               b"spike_count")
        if not p:
            raise RuntimeError(self.ng.GetErrorMessage())
        return np.ctypeslib.as_array(p, (self.neuron.n,))

    def __del__(self):
        try:
            self.ng.ResetKernel()
            _free.append((self.ng, self.lib))
        except Exception:       # at the interpreter's end
            pass


# ---------------------------------------------------------------------
# the networks
# ---------------------------------------------------------------------
UNIFORM_DELAY = {"distribution": "uniform", "low": 0.1, "high": 2.0,
                 "step": 0.1}


def _start(ng, seed):
    ng.ResetKernel()
    ng.SetVerbosityLevel(0)
    ng.SetRandomSeed(seed)


def _v0(case, seed):
    return np.random.default_rng(seed).uniform(
        -70.0, -55.0, case["n"]).astype(np.float32)


def _adex_weights(case):
    """(E, I, Poisson) weights in units of 1/256 nS: those of the 1000-input
    networks, the recurrent ones scaled to the case's in-degree."""
    f = 1000.0 / case["k"] if case["active"] else 1.0
    if case["active"]:
        return max(1, round(13 * f)), max(1, round(90 * f)), 95
    return 13, 64, 26


def _adex(ng, case, seed):
    """aeif_cond_beta neurons, 2 ports, 80 % excitatory, fixed in-degree,
    Poisson drive from one generator or one a neuron."""
    _start(ng, seed)
    n, k = case["n"], case["k"]
    n_e = int(round(0.8 * n))
    k_e = int(round(0.8 * k))
    we, wi, wp = _adex_weights(case)
    neuron = ng.Create("aeif_cond_beta", n, 2)
    if case["active"]:
        ng.SetStatus(neuron, {"E_rev": [0.0, -85.0], "tau_decay": [1.0, 1.0],
                              "tau_rise": [1.0, 1.0]})
        delay = {"distribution": "normal_clipped", "mu": 0.5, "sigma": 0.25,
                 "low": 0.1, "high": 1.25}
    else:
        ng.SetStatus(neuron, dict(wl.C1_NEURON))
        ng.SetStatus(neuron, {"V_m": {"array": _v0(case, seed)}})
        delay = UNIFORM_DELAY
    ng.SetStatus(neuron, {"rk5_tol": case["tol"]})
    own = case["gens"] == "own"
    pg = ng.Create("poisson_generator", n if own else 1)
    ng.SetStatus(pg, {"rate": case["rate"]})
    ng.Connect(neuron[0:n_e], neuron, {"rule": "fixed_indegree",
                                       "indegree": k_e},
               {"weight": we * W, "delay": delay, "receptor": 0})
    ng.Connect(neuron[n_e:n], neuron, {"rule": "fixed_indegree",
                                       "indegree": k - k_e},
               {"weight": wi * W, "delay": delay, "receptor": 1})
    ng.Connect(pg, neuron, {"rule": "one_to_one" if own else "all_to_all"},
               {"weight": wp * W, "delay": 0.1, "receptor": 0})
    return neuron


def _psc(ng, case, seed):
    """Current-based (or alpha-conductance) AdEx neurons: random recurrent
    synapses on every port, Poisson drive on port 0."""
    _start(ng, seed)
    n, k, ports = case["n"], case["k"], case["ports"]
    neuron = ng.Create(case["model"], n, ports)
    cond = "cond" in case["model"]
    if cond:
        ng.SetStatus(neuron, {"E_rev": [0.0] * (ports - 1) + [-85.0]})
    ng.SetStatus(neuron, {"tau_syn": [2.0 + q for q in range(ports)],
                          "V_peak": 0.0,
                          "V_m": {"array": _v0(case, seed)}})
    pg = ng.Create("poisson_generator", 1)
    ng.SetStatus(pg, {"rate": case["rate"]})
    w = 0.25 if cond else 4.0
    for q in range(ports):
        kq = max(1, k // ports)
        inhib = q == ports - 1 and not cond
        ng.Connect(neuron, neuron, {"rule": "fixed_indegree", "indegree": kq},
                   {"weight": -w if inhib else w, "delay": UNIFORM_DELAY,
                    "receptor": q})
    ng.Connect(pg, neuron, {"rule": "all_to_all"},
               {"weight": 0.5 if cond else 40.0, "delay": 0.1,
                "receptor": 0})
    return neuron


def _iaf(ng, case, seed):
    """The layered column: 8 populations of iaf_psc_exp neurons, fixed total
    numbers of synapses per pair, whole-pA weights (below full size the
    recurrent ones grow as the in-degrees shrink)."""
    _start(ng, seed)
    rng = np.random.default_rng(seed)
    sizes = [max(20, int(round(n * case["scale"]))) for n in wl.C2_SIZES]
    off = np.concatenate([[0], np.cumsum(sizes)])
    neuron = ng.Create("iaf_psc_exp", int(off[-1]))
    ng.SetStatus(neuron, {"V_m_rel": {"array": rng.uniform(
        0.0, 15.0, int(off[-1])).astype(np.float32)}})
    pg = ng.Create("poisson_generator", 8)
    # one set of connection probabilities for every seed, the benchmark's:
    # the activity of the column depends on them
    bench = np.random.default_rng(2014)
    bench.uniform(0.0, 15.0, sum(wl.C2_SIZES))
    p = bench.uniform(0.01, 0.15, (8, 8))
    pops = [neuron[int(off[j]):int(off[j + 1])] for j in range(8)]
    w = round(88.0 / min(1.0, case["scale"]))
    for j in range(8):
        ng.SetStatus(pg[j:j + 1], {"rate": 8.0 * wl.C2_K_EXT[j]})
        for i in range(8):
            exc = i % 2 == 0
            ng.Connect(
                pops[i], pops[j],
                {"rule": "fixed_total_number",
                 "total_num": max(1, int(round(p[j, i] * sizes[i] *
                                               sizes[j])))},
                {"weight": float(w if exc else -4 * w),
                 "delay": {"distribution": "normal_clipped",
                           "mu": 1.5 if exc else 0.8,
                           "sigma": 0.75 if exc else 0.4, "low": 0.1,
                           "high": 1.0e3},
                 "receptor": 0 if exc else 1})
        ng.Connect(pg[j:j + 1], pops[j], {"rule": "all_to_all"},
                   {"weight": 88.0, "delay": 0.1, "receptor": 0})
    return neuron


def _stdp(ng, case, seed):
    """aeif_cond_alpha neurons with pair-based STDP on the E -> E synapses,
    one Poisson generator a neuron."""
    _start(ng, seed)
    n, k = case["n"], case["k"]
    n_e, k_e = int(round(0.8 * n)), int(round(0.8 * k))
    neuron = ng.Create("aeif_cond_alpha", n, 2)
    exc, inh = neuron[0:n_e], neuron[n_e:n]
    ng.SetStatus(neuron, dict(wl.C3_NEURON))
    ng.SetStatus(neuron, {"V_m": {"array": _v0(case, seed)},
                          "rk5_tol": 1e-3})
    pg = ng.Create("poisson_generator", n)
    ng.SetStatus(pg, {"rate": case["rate"]})
    sg = ng.CreateSynGroup("stdp", dict(wl.C3_STDP))
    w = {"distribution": "uniform", "low": 0.02, "high": 0.06}
    # E -> E by out-degree: the weights read back have one shape
    ng.Connect(exc, exc, {"rule": "fixed_outdegree", "outdegree": k_e},
               {"weight": w, "delay": UNIFORM_DELAY, "receptor": 0,
                "synapse_group": sg})
    ng.Connect(exc, inh, {"rule": "fixed_indegree", "indegree": k_e},
               {"weight": w, "delay": UNIFORM_DELAY, "receptor": 0})
    ng.Connect(inh, neuron, {"rule": "fixed_indegree", "indegree": k - k_e},
               {"weight": 0.25, "delay": UNIFORM_DELAY, "receptor": 1})
    ng.Connect(pg, neuron, {"rule": "one_to_one"},
               {"weight": 77 * W, "delay": 0.1, "receptor": 0})
    return neuron


def _instances(case):
    """Networks of the ensemble: sizes log-uniform, in-degrees, weight
    scales and rates of their own (the same for every seed, as the sizes of
    the outputs follow them), weights in units of 1/256 nS."""
    rng = np.random.default_rng(case["n_lo"])
    out = []
    for x in wl.c4_instances(case["inst"], 6464, case["n_lo"], case["n_hi"]):
        k = min(x["k"], x["n"] // 5)
        sc = float(rng.uniform(0.5, 1.0))
        out.append({"n": x["n"], "k": k, "w_e": round(13 * sc) * W,
                    "w_i": round(64 * sc) * W,
                    "rate": float(np.float32(min(x["rate"], 9000.0)))})
    return out


def _build(ng, case, seed):
    """1 network of n neurons, in-degree k, delays 1-20 steps, calibrated."""
    return _adex(ng, {"active": False, "n": case["n"], "k": case["k"],
                      "rate": 8000.0, "gens": "one", "tol": 1e-3}, seed)


def _script(s, case, seed):
    ng = s.ng
    s.neuron = _adex(ng, dict(case, active=False, gens="own", tol=1e-3), seed)
    cols = min(10, case["n"])
    s.rec = [ng.CreateRecord("", [v] * cols, s.neuron[0:cols].ToList(),
                             [0] * cols) for v in ("V_m", "w")]


def _samples(case, seed):
    """Logged (features, target) samples of RK5 attempts: normalised state,
    step and error features, and a smooth target of them."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    s = np.zeros((n, 8), np.float32)
    s[:, 0] = rng.normal(1.0, 0.6, n)           # (V - E_L) / 10 mV
    s[:, 1] = rng.uniform(0.0, 3.0, n)          # w / 100 pA
    s[:, 2] = rng.uniform(0.0, 6.0, n)          # g_ex
    s[:, 3] = rng.uniform(0.0, 6.0, n)          # g_in
    s[:, 4] = rng.uniform(-6.0, 0.0, n)         # log2 h / dt
    s[:, 5] = rng.uniform(-1.0, 0.5, n)         # log10(err) / 4
    s[:, 6] = (0.8 * s[:, 4] - 1.5 * s[:, 5] - 0.3 * s[:, 0] +
               0.05 * rng.normal(0.0, 1.0, n))
    return s


def _weights0(seed):
    rng = np.random.default_rng(seed + 1)
    w = np.zeros(_first.PROPOSER_N_PARAM, np.float32)
    w[:192] = rng.uniform(-1.0, 1.0, 192)
    w[192:224] = rng.uniform(-0.1, 0.1, 32)
    w[224:1248] = rng.uniform(-0.4, 0.4, 1024)
    w[1248:1280] = rng.uniform(-0.1, 0.1, 32)
    w[1280:1312] = rng.uniform(-0.2, 0.2, 32)
    return w


_NETWORK = {"adex": _adex, "psc": _psc, "iaf": _iaf, "stdp": _stdp}


def prepare(case, seed):
    s = State(case)
    s.seed = seed
    kind = case["kind"]
    if kind in _NETWORK:
        s.neuron = _NETWORK[kind](s.ng, case, seed)
    elif kind == "ensemble":
        inst = _instances(case)
        s.neuron, _, _ = wl.build_ensemble(s.ng, inst, seed=seed,
                                           w_p=26 * W)
    elif kind == "train":
        _start(s.ng, seed)
        s.ng.ProposerSetSamples(_samples(case, seed))
        s.ng.ProposerSetWeights(_weights0(seed))
    if s.neuron is not None:
        i0 = s.neuron.i0
        s.names = s.ng.GetScalVarNames(i0) + s.ng.GetPortVarNames(i0)
        s.ng.ActivateSpikeCount(s.neuron)
        s.ng.Calibrate()
        if case.get("settle", 0.0) > 0.0:
            s.ng.Simulate(case["settle"])
    return s


def run(state):
    s, case, ng = state, state.case, state.ng
    kind = case["kind"]
    if kind == "train":
        loss = ng.ProposerTrain(case["iters"], batch=case["batch"])
        return {"weights": ng.ProposerGetWeights(), "loss": loss}
    if kind == "build":
        s.neuron = _build(ng, case, s.seed)
        ng.Calibrate()
        got = ng.GetConnectionCounts(s.neuron, n_delay=20)
        return [got["in_degree"], got["out_degree"], got["delay_count"]]
    if kind == "script":
        _script(s, case, s.seed)
        ng.Simulate(case["ms"])
        return [ng.GetRecordDataArray(r) for r in s.rec]
    ng.Simulate(case["ms"])
    out = s.variables()
    out["spikes"] = s.counts()
    if kind == "stdp":
        # the plastic weights of some neurons, as a program follows them
        out["weights"] = ng.GetConnectionArrays(
            source=s.neuron[0:32],
            target=s.neuron[0:int(round(0.8 * case["n"]))])["weight"]
    return out


# ---------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------
def _network_work(n, k, rate, ms, bytes_per, flops_per):
    """Neuron-steps (state read and written) and synaptic events (9 B: the
    target and port, the weight, the event's share of its delay)."""
    steps = ms / DT
    events = rate * 1e-3 * ms * n * k
    return {"bytes": n * steps * bytes_per + 9.0 * events,
            "flops": n * steps * flops_per + 2.0 * events}


def work(case):
    kind = case["kind"]
    if kind == "train":
        m = float(case["iters"]) * case["batch"]
        return {"bytes": 28.0 * m, "flops": 6.0 * 1248.0 * m}
    if kind == "build":
        m = float(case["n"]) * case["k"]
        return {"bytes": 8.0 * m + 84.0 * case["n"], "flops": 0.0}
    if kind in ("script", "adex"):
        act = case.get("active", False)
        return _network_work(case["n"], case["k"], 30.0 if act else 0.0,
                             case["ms"], 72.0, 580.0 if act else 512.0)
    if kind == "psc":
        return _network_work(case["n"], case["k"], 0.0, case["ms"],
                             40.0 + 16.0 * case["ports"],
                             300.0 + 100.0 * case["ports"])
    if kind == "iaf":
        n = 77169 * case["scale"]
        return _network_work(n, 7700.0 * case["scale"], 430.0, case["ms"],
                             40.0, 12.0)
    if kind == "stdp":
        return _network_work(case["n"], case["k"], 4.0, case["ms"], 72.0,
                             515.0)
    n = float(sum(x["n"] for x in _instances(case)))
    return _network_work(n, 550.0, 0.0, case["ms"], 72.0, 512.0)


def tolerance(case):
    kind = case["kind"]
    if kind == "train":
        # 32-bit sums of a minibatch in any order, through the optimiser
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "build":
        return "exact"
    if kind == "stdp":
        # the order of the float additions of the plastic weights moves a
        # spike by a step here and there
        return {"rel": 2e-3, "max": 0.9, "differ": 1e-3}
    if kind in ("script", "ensemble") or (kind == "adex" and
                                          not case["active"]):
        # no recurrent input: the error of the 32-bit step sequence
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}
    # sums exact in any order, so spikes and state are those of one
    # sequence of 32-bit operations; another sequence would give another
    # (equally valid) chaotic trajectory that no tolerance compares
    return "exact"


# ---------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------
_M32 = 0xFFFFFFFF


def _threefry(c0, c1, k0, k1):
    """Word 0 of Threefry2x32-20 (counter tensor c0 and scalar c1)."""
    ks = (k0, k1, 0x1BD11BDA ^ k0 ^ k1)
    x0 = (c0 + ks[0]) & _M32
    x1 = torch.full_like(c0, (c1 + ks[1]) & _M32)
    rot = (13, 15, 26, 6, 17, 29, 16, 24)
    for r in range(20):
        x0 = (x0 + x1) & _M32
        d = rot[r & 7]
        x1 = (((x1 << d) | (x1 >> (32 - d))) & _M32) ^ x0
        if r & 3 == 3:
            s = (r + 1) >> 2
            x0 = (x0 + ks[s % 3]) & _M32
            x1 = (x1 + ks[(s + 1) % 3] + s) & _M32
    return x0


def _thresholds(rate):
    """Poisson CDF of rate * dt as 32-bit thresholds."""
    lam = float(np.float32(_f32(DT) / 1000.0) * np.float32(rate))
    p = math.exp(-lam)
    cdf, k = p, 0
    tab = []
    while cdf * 4294967296.0 < 4294967295.0 and k < 255:
        tab.append(max(0.0, math.ceil(cdf * 4294967296.0) - 1.0))
        k += 1
        p *= lam / k
        cdf += p
    return tab


_CK = ((0.2,), (3 / 40, 9 / 40), (0.3, -0.9, 1.2),
       (-11 / 54, 2.5, -70 / 27, 35 / 27),
       (1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096))
_C5 = (37 / 378, 0.0, 250 / 621, 125 / 594, 0.0, 512 / 1771)
_C4 = (2825 / 27648, 0.0, 18575 / 48384, 13525 / 55296, 277 / 14336, 0.25)


def _f32(x):
    return float(np.float32(x))


def _silent_adex(v0, rates, w_p, seed, steps, device, tol=1e-3, keep=0):
    """State of neurons that never spike (None if one does): adaptive
    Cash-Karp RK5 in 64 bits of the AdEx equations with two beta
    conductances under Poisson input, after `steps` steps and the input of
    the last; with `keep` the (V, w) rows of the first `keep` neurons at
    every step.  rates: (number of neurons, rate) per generator."""
    P = {k: ([_f32(x) for x in v] if isinstance(v, list) else _f32(v))
         for k, v in wl.C1_NEURON.items()}
    f64 = dict(dtype=torch.float64, device=device)
    n = len(v0)
    dt = _f32(DT)
    eps, h_min = _f32(tol), _f32(np.float32(1e-3) * np.float32(DT))
    y = torch.zeros(6, n, **f64)
    y[0] = torch.from_numpy(v0).to(**f64)
    h = torch.full((n,), _f32(np.float32(1e-2) * np.float32(DT)), **f64)
    td, tr = P["tau_decay"], P["tau_rise"]
    tp = td[0] * tr[0] * math.log(td[0] / tr[0]) / (td[0] - tr[0])
    g0 = (1 / tr[0] - 1 / td[0]) / (math.exp(-tp / td[0]) -
                                    math.exp(-tp / tr[0]))
    j = torch.arange(n, dtype=torch.int64, device=device)
    edges = [torch.tensor(_thresholds(r), **f64) for _, r in rates]
    lo = np.concatenate([[0], np.cumsum([m for m, _ in rates])])

    def rhs(z):
        V = torch.clamp(z[0], max=0.0)     # V_peak
        spike = P["Delta_T"] * torch.exp((V - P["V_th"]) / P["Delta_T"])
        syn = z[2] * (P["E_rev"][0] - V) + z[4] * (P["E_rev"][1] - V)
        dV = (-P["g_L"] * ((V - P["E_L"]) - spike) + syn - z[1]) / P["C_m"]
        dw = (P["a"] * (V - P["E_L"]) - z[1]) / P["tau_w"]
        return torch.stack([dV, dw, z[3] - z[2] / td[0], -z[3] / tr[0],
                            z[5] - z[4] / td[1], -z[5] / tr[1]])

    def drive(step):               # the Poisson counts of that step
        u = _threefry(j, step, (seed & _M32) ^ 0x504F4953,
                      (seed >> 32) & _M32).to(torch.float64)
        for g in range(len(rates)):
            part = slice(int(lo[g]), int(lo[g + 1]))
            # counts: thresholds below the draw
            y[3, part] += g0 * w_p * torch.bucketize(u[part], edges[g])

    rows = []
    for step in range(1, steps + 1):
        if step > 1:
            drive(step - 1)
        x = torch.zeros(n, **f64)
        live = j
        fresh = True
        while live.numel():
            z = y[:, live] if live.numel() < n else y
            hl, xl = h[live], x[live]
            if fresh:
                k1 = rhs(z)
                scale = z.abs() + (k1 * hl).abs() + 0.1
            hh = torch.clamp(torch.minimum(hl, dt - xl), min=h_min)
            ks = [k1]
            for a in _CK:
                ks.append(rhs(z + hh * sum(c * q for c, q in zip(a, ks))))
            zn = z + hh * sum(c * q for c, q in zip(_C5, ks) if c)
            err = ((hh * sum((c - d) * q for c, d, q in
                             zip(_C5, _C4, ks))).abs() / scale).amax(0) / eps
            ok = (err <= 1.0) | (hh <= h_min * (1.0 + 1e-5))
            grow = torch.where(err > 1.889568e-4,
                               0.9 * err.clamp(min=1e-30) ** -0.2,
                               torch.full_like(err, 5.0))
            shrink = torch.clamp(0.9 * err.clamp(min=1e-30) ** -0.25,
                                 min=0.1)
            h[live] = hh * torch.where(ok, grow, shrink)
            y[:, live] = torch.where(ok, zn, z)
            x[live] = torch.where(ok, xl + hh, xl)
            if bool((y[0] >= 0.0).any()):
                return None
            # a rejected step keeps its first stage and scale
            again = ~ok
            going = x[live] < dt - h_min
            if bool((again & going).any()):
                # retries and new steps of the same round: the first stage
                # is the same function of the same state, only the scale
                # is kept for the retries
                k1n = rhs(y[:, live])
                sc = y[:, live].abs() + (k1n * h[live]).abs() + 0.1
                scale = torch.where(again, scale, sc)[:, going]
                k1 = torch.where(again, k1, k1n)[:, going]
                fresh = False
            else:
                fresh = True
            live = live[going]
        if keep:
            rows.append(y[:2, :keep].cpu().numpy().copy())
    if keep:
        return rows
    drive(steps)
    y = y.T.cpu().numpy()
    return {"V_m": y[:, 0:1], "w": y[:, 1:2], "g": y[:, [2, 4]],
            "g1": y[:, [3, 5]], "spikes": None}


def _philox(c, k0, k1):
    """Word 0 of Philox4x32-10 on counter columns c (numpy uint64)."""
    c = [x.astype(np.uint64) & np.uint64(_M32) for x in c]
    for _ in range(10):
        p0 = c[0] * np.uint64(0xD2511F53)
        p1 = c[2] * np.uint64(0xCD9E8D57)
        s, m = np.uint64(32), np.uint64(_M32)
        c = [(p1 >> s) ^ c[1] ^ np.uint64(k0), p1 & m,
             (p0 >> s) ^ c[3] ^ np.uint64(k1), p0 & m]
        k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
    return c[0]


def _train(case, seed, device):
    """Adam on the 6-32-32-1 ReLU network, squared error, in 64 bits."""
    s = torch.from_numpy(_samples(case, seed)).double().to(device)
    w = torch.from_numpy(_weights0(seed)).double().to(device)
    m, v = torch.zeros_like(w), torch.zeros_like(w)
    b = np.arange(case["batch"], dtype=np.uint64)
    one = np.ones_like(b)
    loss = 0.0
    for it in range(case["iters"]):
        word = [_philox([b, one * it, one * 0x70726F70, one * q],
                        seed & _M32, 0x74726169) for q in (0, 1)]
        idx = ((word[1] << np.uint64(32)) | word[0]) % np.uint64(case["n"])
        q = s[torch.from_numpy(idx.astype(np.int64)).to(device)]
        W = w.clone().requires_grad_(True)
        h1 = torch.relu(q[:, :6] @ W[:192].reshape(32, 6).T + W[192:224])
        h2 = torch.relu(h1 @ W[224:1248].reshape(32, 32).T + W[1248:1280])
        out = h2 @ W[1280:1312] + W[1312]
        loss = (0.5 * (out - q[:, 6]) ** 2).mean()
        g, = torch.autograd.grad(loss, W)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        w = w - 1e-3 * (m / (1 - 0.9 ** (it + 1))) / (
            (v / (1 - 0.999 ** (it + 1))).sqrt() + 1e-8)
    return {"weights": w.cpu().numpy(), "loss": float(loss)}


def exact(case, seed):
    """64-bit results of the training and of the networks that do not
    spike.  A spiking recurrent network is chaotic: any change of rounding
    moves a spike within some milliseconds, and there is no 64-bit value of
    its trajectory to hold a 32-bit one against; the construction's outputs
    are whole numbers."""
    device = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind == "train":
        return _train(case, seed, device)
    steps = int(round(case.get("ms", 0.0) / DT))
    if kind == "script":
        rows = _silent_adex(_v0(case, seed), [(case["n"], case["rate"])],
                            26 * W, seed, steps, device,
                            keep=min(10, case["n"]))
        if rows is None:
            return None
        cols = min(10, case["n"])
        first = np.stack([_v0(case, seed)[:cols].astype(np.float64),
                          np.zeros(cols)])
        rows = np.stack([first] + rows)
        t = _f32(DT) * np.arange(steps + 1)
        return [np.column_stack([t, rows[:, q]]) for q in (0, 1)]
    if kind == "adex" and not case["active"] and case["n"] * steps <= 2e9:
        return _silent_adex(_v0(case, seed), [(case["n"], case["rate"])],
                            26 * W, seed, steps, device, tol=case["tol"])
    if kind == "ensemble":
        inst = _instances(case)
        n = sum(x["n"] for x in inst)
        v0 = np.random.default_rng(seed).uniform(-70.0, -55.0,
                                                 n).astype(np.float32)
        return _silent_adex(v0, [(x["n"], x["rate"]) for x in inst], 26 * W,
                            seed, steps, device)
    return None
