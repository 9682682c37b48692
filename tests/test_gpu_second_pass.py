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


def run(ngpu, sp, settings):
    groups, _ = wl.build_from_spec(ngpu, sp)
    ngpu.SetKernelStatus(settings)
    ngpu.ActivateSpikeCount(groups[0])
    ngpu.Simulate(60.0)
    out = [np.array(ngpu.GetNeuronVar(0, N, v))
           for v in ("V_m", "w", "g", "g1")]
    out.append(np.array(ngpu.GetNeuronIntVar(0, N, "spike_count")))
    out.append(ngpu.GetHotPathStats())
    return out


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("ports", [1, 2, 3, 4])
def test_second_pass_layouts(ngpu, ports, uniform):
    """Grids of 256 blocks (every list fits the quads), 1 block (64 quads:
    longer lists run on whole waves first), and binned steps, where the pass
    overlaps the next step; 4 ports keep one lane per neuron."""
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
