"""The RK5 updates' lane layouts: neurons on lanes of their own, then one
neuron per quad of lanes for a wave's last neurons.  The second pass of the
AdEx conductance models against the single-pass kernel (one neuron a lane to
the end of the step), the current-based models against the FP32 oracle, bit
for bit.
"""
import numpy as np
import pytest

import netbuild as nb
from neurongpu_amd import workloads as wl

pytestmark = pytest.mark.gpu

N = 700


def spec(ports, uniform, tol=1e-6):
    """Spiking AdEx neurons (drive above the rheobase, refractory for 5
    steps) with recurrent synapses of dyadic weight on every port."""
    rng = np.random.default_rng(10 * ports + uniform)
    I_e = 900.0 if uniform else rng.uniform(500.0, 1500.0, N)
    src = rng.integers(0, N, 20 * N)
    tgt = rng.integers(0, N, 20 * N)
    port = rng.integers(0, ports, 20 * N)
    conns = [{"src": src[port == q], "tgt": tgt[port == q], "weight": 0.25,
              "delay": 0.1 * rng.integers(1, 8, int((port == q).sum())),
              "port": q} for q in range(ports)]
    return {"seed": 3, "conns": conns, "groups": [
        {"model": "aeif_cond_beta", "n": N, "n_port": ports,
         "params": {"I_e": I_e, "t_ref": 0.5,
                    "E_rev": [0.0, -85.0, -10.0, -70.0][:ports],
                    "tau_rise": [0.5, 0.5, 1.0, 2.0][:ports],
                    "tau_decay": [2.0, 5.0, 1.0, 4.0][:ports]},
         "vars": {"V_m": rng.uniform(-70.0, -40.0, N).astype(np.float32)},
         "rk5": {"rk5_tol": tol}}]}


def run(ngpu, sp, settings, ms=60.0, change=()):
    groups, _ = wl.build_from_spec(ngpu, sp)
    for node, name, val in change:
        ngpu.SetStatus([node], {name: val})
    ngpu.SetKernelStatus(settings)
    ngpu.ActivateSpikeCount(groups[0])
    ngpu.Simulate(ms)
    out = [np.array(ngpu.GetNeuronVar(0, N, v))
           for v in ("V_m", "w", "g", "g1")]
    out.append(np.array(ngpu.GetNeuronIntVar(0, N, "spike_count")))
    out.append(ngpu.GetHotPathStats())
    return out


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ports", [1, 2, 3, 4])
def test_second_pass_layouts(ngpu, ports, uniform):
    """Up to 3 ports these steps run in one launch (whatever the budget and
    the second pass's grid), and binned, where the pass overlaps the next
    step; 4 ports run in two passes, with one lane per neuron."""
    print("case second_pass", ports, uniform, flush=True)
    sp = spec(ports, uniform)
    want = run(ngpu, sp, {"rk5_two_pass": 0})
    assert want[4].sum() > 2 * N
    for st in ({"rk5_pass2_grid": 256}, {"rk5_pass2_grid": 1},
               {"rk5_pass2_grid": 1, "rk5_budget": 3},
               {"delivery_mode": 1}, {"delivery_mode": 1,
                                      "rk5_pass2_grid": 1}):
        print("  settings", st, flush=True)
        got = run(ngpu, sp, st)
        for a, b in zip(want[:5], got[:5]):
            assert np.array_equal(a, b)
        # the same attempts, accepted and rejected
        assert got[5] == want[5]


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ports", [1, 2, 3])
def test_second_pass_of_a_large_network(ngpu, ports, uniform):
    """The second pass in the launch of the delivery, as networks of more
    than 65536 neurons run it (here with silent ones beside the spiking):
    256 blocks (every list fits the quads), 1 block (64 quads; in the first
    step, which starts at a hundredth of the time step, all 700 neurons are
    listed and run on whole waves first), a budget of 3 attempts."""
    print("case second_pass_large", ports, uniform, flush=True)
    sp = spec(ports, uniform)
    sp["groups"].append({"model": "iaf_psc_exp", "n": 65536})
    want = run(ngpu, sp, {"rk5_two_pass": 0, "delivery_mode": 0})
    assert want[4].sum() > 2 * N
    for st in ({"rk5_pass2_grid": 256}, {"rk5_pass2_grid": 1},
               {"rk5_pass2_grid": 256, "rk5_budget": 3},
               {"rk5_pass2_grid": 1, "rk5_budget": 3}):
        print("  settings", st, flush=True)
        got = run(ngpu, sp, dict(st, delivery_mode=0))
        for a, b in zip(want[:5], got[:5]):
            assert np.array_equal(a, b)
        assert got[5] == want[5]
        # two launches a step: first pass; second pass with the delivery
        ngpu.SetKernelTiming(1)
        ngpu.Simulate(0.5)
        kinds = ngpu.GetKernelTimes()
        ngpu.SetKernelTiming(0)
        assert kinds["aeif_rk5_pass2"][1] == kinds["aeif_rk5"][1] == 5
        assert "delivery" not in kinds


NAN, INF = float("nan"), float("inf")


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ports", [1, 2, 3])
def test_neurons_with_invalid_state(ngpu, ports, uniform):
    """NaN and infinite membrane potentials, adaptation currents and
    conductances in some neurons of a wave: the same bits (any NaN as NaN),
    attempts and forced accepts in every form of the step."""
    print("case invalid_state", ports, uniform, flush=True)
    sp = spec(ports, uniform)
    odd = [(3, "V_m", NAN), (70, "w", NAN), (71, "g", [NAN] * ports),
           (72, "g1", [NAN] * ports), (200, "V_m", INF),
           (201, "V_m", -INF), (264, "w", INF), (265, "w", -INF),
           (266, "g", [INF] * ports), (267, "g1", [INF] * ports),
           (N - 1, "g1", [0.0] * (ports - 1) + [NAN])]
    want = run(ngpu, sp, {"rk5_two_pass": 0}, 5.0, odd)
    assert np.isnan(want[0][[3, 72, N - 1]]).all()
    for st in ({}, {"fuse_delivery": 0}, {"delivery_mode": 1}):
        print("  settings", st, flush=True)
        got = run(ngpu, sp, st, 5.0, odd)
        for a, b in zip(want[:4], got[:4]):
            assert np.array_equal(a, b, equal_nan=True)
        assert np.array_equal(want[4], got[4])
        assert got[5] == want[5]


@pytest.mark.parametrize("ports", [1, 2, 3])
def test_attempt_cap(ngpu, ports):
    """A neuron whose error is NaN at a minimum step of 1e-6 time steps
    reaches the cap of attempts and gives the time step up."""
    print("case attempt_cap", ports, flush=True)
    sp = spec(ports, True)
    sp["groups"][0]["rk5"]["h_min_rel"] = 1e-6
    odd = [(i, "g1", [0.0] * (ports - 1) + [NAN]) for i in (5, 300, N - 1)]
    want = run(ngpu, sp, {"rk5_two_pass": 0}, 0.3, odd)
    assert want[5]["rk5_rejected"] > 3 * 3 * 40000
    assert want[5]["rk5_accepted"] < 3 * 3 * 60000 + 3 * N * 100
    for st in ({}, {"fuse_delivery": 0}, {"delivery_mode": 1}):
        print("  settings", st, flush=True)
        got = run(ngpu, sp, st, 0.3, odd)
        for a, b in zip(want[:4], got[:4]):
            assert np.array_equal(a, b, equal_nan=True)
        assert np.array_equal(want[4], got[4])
        assert got[5] == want[5]


@pytest.mark.parametrize("h_min", [1e-3, 1e-6])
@pytest.mark.parametrize("ports", [1, 3])
@pytest.mark.parametrize("model", ["aeif_psc_alpha", "aeif_psc_exp"])
def test_psc_neurons_with_invalid_state(ngpu, model, ports, h_min):
    """The same for the current-based models against the FP32 oracle; at the
    smaller minimum step the NaN errors reach the cap."""
    print("case psc_invalid", model, ports, h_min, flush=True)
    n, steps = 70, (30 if h_min == 1e-3 else 2)
    rng = np.random.default_rng(ports)
    last = "I1_syn" if model == "aeif_psc_alpha" else "I_syn"
    sp = {"seed": 7, "groups": [
        {"model": model, "n": n, "n_port": ports,
         "params": {"I_e": rng.uniform(700.0, 1500.0, n), "t_ref": 0.5,
                    "V_peak": 0.0},
         "vars": {"V_m": rng.uniform(-70.0, -50.0, n).astype(np.float32)},
         "rk5": {"h_min_rel": h_min}}]}
    odd = [(5, last, NAN), (66, last, NAN)]
    if h_min == 1e-3:
        odd += [(0, "V_m", NAN), (1, "w", NAN), (2, "I_syn", INF),
                (63, "V_m", INF), (64, "V_m", -INF), (65, "w", INF),
                (67, "w", -INF), (68, last, -INF)]
    groups, _ = nb.build_engine(ngpu, sp)
    net, og = nb.build_oracle(sp, "f32")
    for name in {v for _, v, _ in odd}:
        vals = np.array(og[0].get(name), dtype=np.float64)
        for i, v, x in odd:
            if v == name:
                vals[i] = x
                ngpu.SetStatus([i], {v: x if v in ("V_m", "w")
                                     else [x] * ports})
        og[0].set(name, vals)
    ngpu.ActivateSpikeCount(groups[0])
    ngpu.Simulate(0.1 * steps)
    net.run(steps)
    for v in ("V_m", "w"):
        assert np.array_equal(np.array(ngpu.GetNeuronVar(0, n, v)),
                              np.array(og[0].get(v), dtype=np.float32),
                              equal_nan=True)
    cur = np.array(ngpu.GetNeuronVar(0, n, "I_syn"))
    for q in range(ports):
        assert np.array_equal(cur.reshape(n, ports)[:, q],
                              np.array(og[0].get("I_syn", q),
                                       dtype=np.float32), equal_nan=True)
    count = np.array(ngpu.GetNeuronIntVar(0, n, "spike_count"))
    _, node, times = net.spikes()
    want = np.zeros(n, int)
    np.add.at(want, np.asarray(node, int), np.asarray(times, int))
    assert np.array_equal(count, want)


@pytest.mark.parametrize("n", [1, 70, 300])
@pytest.mark.parametrize("ports", [1, 2, 3, 4])
@pytest.mark.parametrize("model", ["aeif_psc_alpha", "aeif_psc_exp"])
def test_psc_layouts(ngpu, model, ports, n):
    """1 neuron (quads from the start), a whole wave and some lanes, several
    blocks; 4 ports keep one lane per neuron.  Delta_T = 0 in the largest."""
    print("case psc_layouts", model, ports, n, flush=True)
    rng = np.random.default_rng(100 * ports + n)
    m = 10 * n
    conns = [{"src": rng.integers(0, n, m), "tgt": rng.integers(0, n, m),
              "weight": 8.0 * rng.integers(-2, 5, m),
              "delay": 0.1 * rng.integers(1, 8, m), "port": q}
             for q in range(ports)]
    params = {"I_e": rng.uniform(700.0, 1500.0, n), "t_ref": 0.5,
              "V_peak": 0.0, "tau_syn": [2.0, 1.0, 5.0, 3.0][:ports]}
    if n == 300:
        params["Delta_T"] = np.where(np.arange(n) % 5 == 0, 0.0, 2.0)
    sp = {"seed": 7, "conns": conns, "groups": [
        {"model": model, "n": n, "n_port": ports, "params": params,
         "vars": {"V_m": rng.uniform(-70.0, -50.0, n).astype(np.float32)}}],
        "records": [(i, v, 0) for i in (0, n // 2, n - 1)
                    for v in ("V_m", "w")]}
    groups, recs = nb.build_engine(ngpu, sp)
    ngpu.ActivateSpikeCount(groups[0])
    ngpu.Simulate(50.0)
    net, _ = nb.build_oracle(sp, "f32")
    net.run(500)
    orc = net.records()
    for k, r in enumerate(recs):
        data = ngpu.GetRecordDataArray(r)
        assert np.array_equal(orc[:, 1 + k].astype(np.float32), data[:, 1])
    count = np.array(ngpu.GetNeuronIntVar(0, n, "spike_count"))
    _, node, times = net.spikes()
    want = np.zeros(n, int)
    np.add.at(want, np.asarray(node, int), np.asarray(times, int))
    assert np.array_equal(count, want) and count.sum() > 0


def test_switches_between_step_forms(ngpu):
    """Two AdEx groups and an iaf_psc_exp group coupled by dyadic synapses:
    steps in one launch, in two passes and binned with overlap, switched
    between and within Simulate calls, against single-pass steps."""
    print("case step_forms", flush=True)
    rng = np.random.default_rng(17)
    n = [300, 200, 150]
    off = [0, 300, 500]
    conns = []
    for s in range(3):
        for t in range(3):
            m = 4000
            conns.append({"src": off[s] + rng.integers(0, n[s], m),
                          "tgt": off[t] + rng.integers(0, n[t], m),
                          "weight": 0.25 if t < 2 else 16.0,
                          "delay": 0.1 * rng.integers(1, 12, m), "port": 0})
    sp = {"seed": 5, "conns": conns, "groups": [
        {"model": "aeif_cond_beta", "n": n[0], "n_port": 2,
         "params": {"I_e": 800.0, "t_ref": 0.3},
         "vars": {"V_m": rng.uniform(-70., -40., n[0]).astype(np.float32)}},
        {"model": "aeif_cond_alpha", "n": n[1], "n_port": 1,
         "params": {"I_e": rng.uniform(600.0, 900.0, n[1])}},
        {"model": "iaf_psc_exp", "n": n[2], "params": {"I_e": 500.0}}]}

    def go(phases):
        groups, _ = wl.build_from_spec(ngpu, sp)
        for g in groups:
            ngpu.ActivateSpikeCount(g)
        out = []
        for st in phases:
            ngpu.SetKernelStatus(st)
            ngpu.SetSimTime(7.0)
            ngpu.StartSimulation()
            for k in range(70):
                if k == 35 and st.get("delivery_mode") == 1:
                    ngpu.SetKernelStatus("delivery_mode", 0)
                ngpu.SimulationStep()
            ngpu.EndSimulation()
            out += [np.array(ngpu.GetNeuronVar(g.i0, g.n, v)) for g, v in
                    zip(groups, ("V_m", "g1", "V_m_rel"))]
            out += [np.array(ngpu.GetNeuronIntVar(g.i0, g.n, "spike_count"))
                    for g in groups]
        return out

    one = {"rk5_two_pass": 1, "fuse_delivery": 1, "delivery_mode": 0}
    two = dict(one, fuse_delivery=0)
    bins = dict(one, delivery_mode=1)
    want = go([dict(one, rk5_two_pass=0)] * 7)
    got = go([one, two, one, bins, one, bins, two])
    assert want[-1].sum() > 0 and want[-3].sum() > 0
    for a, b in zip(want, got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("settings", [{"fuse_delivery": 0},
                                      {"delivery_mode": 1}])
@pytest.mark.parametrize("lengths", [(9, 1, 9), (10, 2, 8), (11, 3, 7),
                                     (9, 36, 12)])
def test_two_pass_switched_off_and_on(ngpu, settings, lengths):
    """rk5_two_pass 1, 0, 1 between steps of one run, the single-pass steps
    of every length modulo the four sets of lists, with second passes that
    end their step and with overlapped ones: as in single-pass steps alone."""
    print("case two_pass_switch", settings, lengths, flush=True)
    sp = spec(2, True)

    def go(passes):
        groups, _ = wl.build_from_spec(ngpu, sp)
        ngpu.SetKernelStatus(settings)
        ngpu.ActivateSpikeCount(groups[0])
        ngpu.SetSimTime(0.1 * sum(lengths) * 6)
        ngpu.StartSimulation()
        for _ in range(6):
            for on, steps in zip(passes, lengths):
                ngpu.SetKernelStatus("rk5_two_pass", on)
                for _ in range(steps):
                    ngpu.SimulationStep()
        ngpu.EndSimulation()
        out = [np.array(ngpu.GetNeuronVar(0, N, v))
               for v in ("V_m", "w", "g", "g1")]
        out.append(np.array(ngpu.GetNeuronIntVar(0, N, "spike_count")))
        return out, ngpu.GetHotPathStats()

    want, st_want = go((0, 0, 0))
    got, st_got = go((1, 0, 1))
    assert want[4].sum() > 0
    for a, b in zip(want, got):
        assert np.array_equal(a, b)
    assert st_got["syn_events"] == st_want["syn_events"]
    assert st_got["rk5_accepted"] == st_want["rk5_accepted"]
    assert st_got["rk5_rejected"] == st_want["rk5_rejected"]
