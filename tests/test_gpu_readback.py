"""Reads of the state by node ranges and lists, the refractory count (the one
parameter row the device writes) and plastic weights by source range, which
copies only that range once the network runs.
"""
import numpy as np
import pytest

from neurongpu_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,ports", [("aeif_cond_beta", 2),
                                         ("aeif_psc_exp", 3),
                                         ("izhikevich_cond_beta", 1),
                                         ("iaf_psc_exp", 1)])
def test_range_and_list_reads(ngpu, model, ports):
    print("case readback", model, flush=True)
    n = 5000
    ngpu.ResetKernel()
    ngpu.SetVerbosityLevel(0)
    ns = ngpu.Create(model, n, ports)
    ngpu.SetStatus(ns, {"I_e": 900.0 if model.startswith("aeif") else
                        30.0 if model.startswith("izh") else 700.0,
                        "t_ref": 1.5})
    v = "V_m_rel" if model == "iaf_psc_exp" else "V_m"
    ngpu.SetStatus(ns, {v: {"array": np.linspace(-69.0, -55.0, n)
                            .astype(np.float32)}})
    ngpu.ActivateSpikeCount(ns)
    seen = 0
    for _ in range(4):
        ngpu.Simulate(20.0)
        nodes = [0, 1, 4095, 4096, n - 1]
        for name in ngpu.GetScalVarNames(0) + ngpu.GetPortVarNames(0):
            whole = ngpu.GetNeuronVar(0, n, name)
            assert [whole[i] for i in nodes] == ngpu.GetNeuronPtVar(nodes,
                                                                    name)
            assert whole[4090:4100] == ngpu.GetNeuronVar(4090, 10, name)
        for name in ngpu.GetScalParamNames(0):
            whole = ngpu.GetNeuronParam(0, n, name)
            assert [whole[i] for i in nodes] == ngpu.GetNeuronPtParam(nodes,
                                                                      name)
            if name == "refractory_step":
                seen += int(np.count_nonzero(whole))
        c = ngpu.GetNeuronIntVar(0, n, "spike_count")
        assert [c[i] for i in nodes] == ngpu.GetNeuronPtIntVar(
            nodes, "spike_count")
    assert sum(c) > 0
    if model != "iaf_psc_exp":
        assert seen > 0      # some neuron was refractory at a read


# parameters with a value per neuron, and per port and half of the neurons
SCAL = {"aeif_cond_beta": ["C_m", "den_delay"],
        "aeif_psc_exp": ["C_m", "V_peak"],
        "izhikevich_cond_beta": ["a", "d"]}
PORT = {"aeif_cond_beta": {"E_rev": (0.0, -85.0), "tau_decay": (2.0, 5.0)},
        "aeif_psc_exp": {"tau_syn": (2.0, 1.0, 5.0)},
        "izhikevich_cond_beta": {"tau_rise": (1.5,), "E_rev": (-3.0,)}}
DRIVE = {"aeif_cond_beta": 900.0, "aeif_psc_exp": 900.0,
         "izhikevich_cond_beta": 30.0}


@pytest.mark.parametrize("model", list(SCAL))
def test_refractory_count_and_parameters_by_value(ngpu, model):
    """The refractory count step by step: t_ref / dt after a spike (one less
    where the spike was not in the step's last RK5 step), then one less per
    step; the other parameters as they were set."""
    print("case readback_values", model, flush=True)
    n, R, ports = 5000, 15, len(next(iter(PORT[model].values())))
    ngpu.ResetKernel()
    ngpu.SetVerbosityLevel(0)
    ns = ngpu.Create(model, n, ports)
    ngpu.SetStatus(ns, {"t_ref": 0.1 * R, "I_e": DRIVE[model]})
    ngpu.SetStatus(ns, {"V_m": {"array": np.linspace(-45.0, -65.0, n)
                                .astype(np.float32)}})
    scal = {}
    for k, name in enumerate(SCAL[model]):
        base = np.array(ngpu.GetNeuronParam(0, n, name), dtype=np.float32)
        scal[name] = (base + np.arange(n) % 7 * 0.1).astype(np.float32)
        ngpu.SetStatus(ns, {name: {"array": scal[name]}})
    port = {}
    for name, vals in PORT[model].items():
        other = [v + 0.5 for v in vals]
        ngpu.SetStatus(ns, {name: list(vals)})
        ngpu.SetStatus(ns[n // 2:n], {name: other})
        port[name] = np.repeat([vals, other], n // 2, axis=0)
    ngpu.ActivateSpikeCount(ns)
    ngpu.SetSimTime(25.0)
    ngpu.StartSimulation()
    refr, count = np.zeros(n), np.zeros(n, int)
    at_end = 0
    for step in range(250):
        ngpu.SimulationStep()
        r = np.array(ngpu.GetNeuronParam(0, n, "refractory_step"))
        c = np.array(ngpu.GetNeuronIntVar(0, n, "spike_count"))
        spk = c > count
        assert np.array_equal(r[~spk], np.maximum(refr - 1.0, 0.0)[~spk])
        assert np.isin(r[spk], (R, R - 1)).all()
        at_end += int((r[spk] == R).sum())
        refr, count = r, c
        if step % 50 == 0:
            for name in scal:
                assert np.array_equal(
                    np.array(ngpu.GetNeuronParam(0, n, name),
                             dtype=np.float32), scal[name])
    ngpu.EndSimulation()
    assert count[0] > 0 and count[-1] > 0 and at_end < count.sum()
    for name in ngpu.GetPortParamNames(0):
        whole = np.array(ngpu.GetNeuronParam(0, n, name)).reshape(n, ports)
        nodes = [0, n // 2 - 1, n // 2, 4096, n - 1]
        assert np.array_equal(
            whole[nodes],
            np.array(ngpu.GetNeuronPtParam(nodes, name)).reshape(-1, ports))
        if name in port:
            assert np.array_equal(whole, port[name].astype(np.float32))


def test_plastic_weights_by_source_range(ngpu):
    print("case readback plastic", flush=True)
    sp = wl.c3_spec(0.005, k=50, w_p=0.6)
    wl.build_from_spec(ngpu, sp)
    n_e = sp["populations"][0][1]
    ngpu.Simulate(100.0)
    ns = ngpu.NodeSeq(0, n_e)
    part = [ngpu.GetConnectionArrays(source=ns[i:i + 100], target=ns)
            for i in (0, 300)]
    before = ngpu.GetConnectionArrays(source=ns, target=ns)
    # the same once a whole-store query has made the host copy
    ngpu.GetConnections(ns[0:1], ns)
    for i, p in zip((0, 300), part):
        sel = (before["source"] >= i) & (before["source"] < i + 100)
        for key in p:
            assert np.array_equal(p[key], before[key][sel])
    assert np.all(before["syn"] == 1)
    # and after more steps, when that copy is old
    ngpu.Simulate(100.0)
    part = ngpu.GetConnectionArrays(source=ns[0:100], target=ns)
    after = ngpu.GetConnectionArrays(source=ns, target=ns)
    sel = after["source"] < 100
    for key in part:
        assert np.array_equal(part[key], after[key][sel])
    assert np.any(after["weight"] != before["weight"])


def test_many_plastic_queries(ngpu):
    """One query per source, again after more steps: the first ones read
    their range from the device, the later ones the host copy that they are
    worth by then; both as one query of all sources."""
    print("case readback many", flush=True)
    sp = wl.c3_spec(0.005, k=50, w_p=0.6)
    wl.build_from_spec(ngpu, sp)
    n_e = sp["populations"][0][1]
    ns = ngpu.NodeSeq(0, n_e)
    weights = []
    for _ in range(2):
        ngpu.Simulate(100.0)
        parts = [ngpu.GetConnectionArrays(source=ns[i:i + 1], target=ns)
                 for i in range(n_e)]
        whole = ngpu.GetConnectionArrays(source=ns, target=ns)
        for key in whole:
            assert np.array_equal(whole[key],
                                  np.concatenate([p[key] for p in parts]))
        weights.append(whole["weight"])
    assert np.any(weights[0] != weights[1])
