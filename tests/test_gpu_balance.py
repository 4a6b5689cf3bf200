"""Spikes of neighbours cost what spikes spread over the network cost. Neurons
that fire together are often next to each other (a stimulated population, a
layer), so no path may leave their delivery to the few workgroups or waves that
hold them. Each case times the same network and the same number of forced
neurons in every cycle, adjacent and spread, the best of several runs each:
adjacent ones may take at most twice as long, half as long again on the fused
kernel."""
import time

import numpy as np
import pytest

from parity import hip_sim
from nemosim_amd import examples

pytestmark = pytest.mark.gpu

CYCLES = 20


def best(f, reps=7):
    f()
    times = []
    for _ in range(reps):
        t = time.perf_counter()
        f()
        times.append(time.perf_counter() - t)
    return min(times)


def simulation(nemo_mod, n, m, mode="auto", stdp=False):
    spec = examples.izhikevich_80_20(n, m, seed=n, stdp=stdp)
    net = spec.to_nemo(nemo_mod)
    conf = nemo_mod.Configuration()
    conf.set_write_only_synapses()
    conf.set_step_mode(mode)
    if stdp:
        pre, post = examples.stdp_window()
        conf.set_stdp_function(pre, post, min_e=0.0, max_e=1.0, min_i=0.0, max_i=-1.0)
    return nemo_mod.Simulation(net, conf)


def populations(n, pop):
    return list(range(pop)), (np.arange(pop, dtype=np.int64) * n // pop).tolist()


@pytest.mark.parametrize("stdp", [False, True])
def test_per_cycle_step(nemo_mod, stdp):
    n = 300000
    sim = simulation(nemo_mod, n, 60, stdp=stdp)
    assert sim.info()["fused"] == 0
    adjacent, spread = [best(lambda: sim.run(CYCLES, fstim=[p] * CYCLES)) for p in populations(n, 256)]
    assert adjacent < 2.0 * spread, (adjacent, spread)


@pytest.mark.parametrize("n,m,pop,stdp", [
    (5000, 1000, 1000, False),       # up to 64 words per wave
    (50000, 300, 2000, False),       # up to 256
    (200000, 100, 2000, False),      # more
    (20000, 300, 1000, True),
])
def test_fused(nemo_mod, n, m, pop, stdp):
    sim = simulation(nemo_mod, n, m, stdp=stdp)
    assert sim.info()["fused"] == 1
    adjacent, spread = [best(lambda: sim.run(CYCLES, fstim=[p] * CYCLES)) for p in populations(n, pop)]
    assert adjacent < 1.5 * spread, (adjacent, spread)


@pytest.mark.parametrize("n,m", [(5000, 1000), (50000, 1000)])
def test_step(nemo_mod, n, m):
    """steps with 60 forced neurons, more of which at once take another path"""
    sim = simulation(nemo_mod, n, m)

    def steps(pop):
        for _ in range(CYCLES):
            sim.step(pop)

    adjacent, spread = [best(lambda: steps(p)) for p in populations(n, 60)]
    assert adjacent < 2.0 * spread, (adjacent, spread)


def test_step_long_rows(nemo_mod):
    """steps with four forced neurons with rows of 30000 synapses"""
    n = 100000

    def run(which):
        spec = examples.izhikevich_80_20(n, 20, seed=3)
        length = np.full(n, 20, np.int64)
        length[which] = 30000
        spec.rowptr = np.concatenate([[0], np.cumsum(length)]).astype(np.uint64)
        rng, count = np.random.default_rng(4), int(length.sum())
        spec.targets = rng.integers(0, n, count).astype(np.uint32)
        spec.delays = rng.integers(1, 21, count).astype(np.uint8)
        spec.weights = rng.uniform(-0.1, 0.1, count).astype(np.float32)
        spec.plastic = np.zeros(count, np.uint8)
        sim = hip_sim(nemo_mod, spec)

        def steps():
            for _ in range(CYCLES):
                sim.step(which)

        return best(steps)

    adjacent, spread = [run(p) for p in populations(n, 4)]
    assert adjacent < 2.0 * spread, (adjacent, spread)


def test_per_cycle_step_long_rows(nemo_mod):
    """neurons with rows of 10000 synapses, next to each other and far apart"""
    n, hubs = 270000, 20

    def run(which):
        spec = examples.izhikevich_80_20(n, 20, seed=3)
        length = np.full(n, 20, np.int64)
        length[which] = 10000
        spec.rowptr = np.concatenate([[0], np.cumsum(length)]).astype(np.uint64)
        rng, count = np.random.default_rng(4), int(length.sum())
        spec.targets = rng.integers(0, n, count).astype(np.uint32)
        spec.delays = rng.integers(1, 21, count).astype(np.uint8)
        spec.weights = rng.uniform(-0.1, 0.1, count).astype(np.float32)
        spec.plastic = np.zeros(count, np.uint8)
        sim = hip_sim(nemo_mod, spec)
        assert sim.info()["fused"] == 0
        return best(lambda: sim.run(CYCLES, fstim=[which] * CYCLES))

    adjacent, spread = [run(p) for p in populations(n, hubs)]
    assert adjacent < 2.0 * spread, (adjacent, spread)


@pytest.mark.parametrize("n,m,pop,stdp", [(20000, 300, 600, False), (20000, 300, 128, True)])
def test_plugin_step(nemo_mod, n, m, pop, stdp):
    sim = simulation(nemo_mod, n, m, mode="plugins", stdp=stdp)
    adjacent, spread = [best(lambda: sim.run(CYCLES, fstim=[p] * CYCLES)) for p in populations(n, pop)]
    assert adjacent < 2.0 * spread, (adjacent, spread)
