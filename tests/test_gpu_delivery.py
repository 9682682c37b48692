"""The delivery's event enumeration and the binned scatter at the sizes where
they branch: long and short segments, wave tiles with more events than a
block buffers, blocks that work in rounds, bins beyond their capacity, few
and many delay slots.  Weights and heights are dyadic, so every mode gives
the atomic delivery's sums bit for bit.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def build(ngpu, n, n_src, k, slots, seed):
    """n_src spike generators (one spike each, steps 1-3, heights 1, 2, 0.5)
    with k synapses each onto n iaf_psc_exp neurons on both ports, delays
    over `slots` steps, most of them on one step."""
    rng = np.random.default_rng(seed)
    ngpu.ResetKernel()
    ngpu.SetVerbosityLevel(0)
    neuron = ngpu.Create("iaf_psc_exp", n)
    gen = ngpu.Create("spike_generator", n_src)
    for i in range(n_src):
        ngpu.SetStatus([gen[i]], {
            "spike_times": [0.1 * float(1 + i % 3)],
            "spike_heights": [float([1.0, 2.0, 0.5][i % 3])]})
    m = n_src * k
    src = np.repeat(np.arange(gen.i0, gen.i0 + n_src, dtype=np.int32), k)
    tgt = rng.integers(0, n, m).astype(np.int32)
    d = np.where(rng.random(m) < 0.7, min(3, slots),
                 rng.integers(1, slots + 1, m))
    for port in (0, 1):
        sel = rng.random(m) < 0.5 if port == 0 else ~sel
        ngpu.Connect(src[sel], tgt[sel], {"rule": "one_to_one"}, {
            "weight": {"array": rng.integers(1, 16, int(sel.sum())) * 0.25},
            "delay": {"array": (d[sel] * 0.1).astype(np.float32)},
            "receptor": port})
    return neuron


def state(ngpu, neuron, settings, steps):
    ngpu.SetKernelStatus(settings)
    ngpu.SetSimTime(0.1 * steps)
    ngpu.StartSimulation()
    out = []
    for _ in range(steps):      # the sums of every step, before they decay
        ngpu.SimulationStep()
        out += [np.array(ngpu.GetNeuronVar(neuron.i0, neuron.n, v))
                for v in ("I_syn_ex", "I_syn_in")]
    ngpu.EndSimulation()
    return out


@pytest.mark.parametrize("n,n_src,k,slots", [
    (1000, 1, 1, 1), (1000, 7, 63, 2), (5000, 65, 129, 20),
    (20000, 3, 40000, 5),       # a pair of 28000 events
    (40000, 300, 700, 64), (3000, 90, 500, 65),
    (6000, 2000, 300, 1),       # wave tiles of many pairs, 12000 events
    (9000, 33, 8200, 2)])       # pieces of a pair that end off a multiple
def test_delivery_modes_agree(ngpu, n, n_src, k, slots):
    print("case delivery_modes", n, n_src, k, slots, flush=True)
    steps = min(slots, 12) + 6
    want = None
    for st in ({"delivery_mode": 0}, {"delivery_mode": 0, "delivery_grid": 1,
                                      "delivery_tile_max": 64},
               {"delivery_mode": 1},
               # 2 blocks: 16 waves take every pair, in rounds
               {"delivery_mode": 1, "delivery_grid": 1},
               {"delivery_mode": 1, "delivery_bin_capacity": 1000},
               {"delivery_mode": 3},
               {"delivery_mode": 3, "delivery_tile_shift": 10,
                "delivery_tile_split": 2}):
        print("  settings", st, flush=True)
        neuron = build(ngpu, n, n_src, k, slots, 5 * n + k)
        got = state(ngpu, neuron, st, steps)
        if want is None:
            want = got
            assert sum(float(np.abs(w).sum()) for w in want) > 0.0
        for a, b in zip(want, got):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("targets", [100000, 3000])
def test_binned_buffer_holds_the_synapses(ngpu, targets):
    """1e7 synapses onto 25 accumulator ranges, evenly or (3000 targets) all
    onto the first ranges of the two ports: the buffer of the binned mode
    takes 8 bytes a synapse, and the sums are the atomic delivery's."""
    print("case binned_buffer", targets, flush=True)
    n, n_src, k = 100000, 100, 50000

    def go(mode):
        ngpu.ResetKernel()
        ngpu.SetVerbosityLevel(0)
        neuron = ngpu.Create("iaf_psc_exp", n)
        gen = ngpu.Create("spike_generator", n_src)
        for i in range(n_src):
            ngpu.SetStatus([gen[i]], {"spike_times": [0.1 * (1 + i % 4)]})
        for port in (0, 1):
            ngpu.Connect(gen, ngpu.NodeSeq(neuron.i0, targets),
                         {"rule": "fixed_total_number", "total_num": n_src * k},
                         {"weight": 0.25, "delay": 0.2, "receptor": port})
        ngpu.SetKernelStatus("delivery_mode", mode)
        ngpu.SetSimTime(0.8)
        ngpu.StartSimulation()
        free = torch.cuda.mem_get_info()[0]
        ngpu.SimulationStep()
        used = free - torch.cuda.mem_get_info()[0]
        for _ in range(7):
            ngpu.SimulationStep()
        ngpu.EndSimulation()
        return used, [np.array(ngpu.GetNeuronVar(neuron.i0, n, v))
                      for v in ("I_syn_ex", "I_syn_in")]

    _, want = go(0)
    used, got = go(1)
    assert used < 8 * 2 * n_src * k + (64 << 20)
    for a, b in zip(want, got):
        assert a.any() and np.array_equal(a, b)
