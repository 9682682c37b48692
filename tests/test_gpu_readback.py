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
