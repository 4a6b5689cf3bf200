"""Kuramoto networks whose rows differ greatly in length (hubs), which are
shared between workgroups by couplings: bit for bit against the oracle, with
hubs at both ends and in the middle, one row that holds everything, empty rows
around it, and networks whose shares take one to four rounds of the search; and
hubs next to each other take no longer than hubs far apart."""
import time

import numpy as np
import pytest

from test_gpu_kuramoto import Pair

pytestmark = pytest.mark.gpu


def degrees(n, mean, hubs):
    """about `mean` couplings each (0 to 2 mean), and hubs {index: couplings}"""
    deg = np.random.default_rng(n).integers(0, 2 * mean + 1, n)
    for i, d in hubs.items():
        deg[i] = d
    return deg


def network(deg, seed):
    rng = np.random.default_rng(seed)
    n, count = len(deg), int(deg.sum())
    tgt = np.repeat(np.arange(n), deg)
    src = rng.integers(0, n, count)
    order = np.argsort(src, kind="stable")
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.uint64)
    return (rowptr, tgt[order].astype(np.uint32), rng.integers(1, 32, count).astype(np.uint8),
            rng.normal(0.0, 0.02, count).astype(np.float32))


@pytest.mark.parametrize("deg", [
    degrees(1025, 3, {0: 3000, 1024: 5000}),
    degrees(3000, 0, {1500: 9000}),                          # everything in one row
    degrees(4097, 4, {i: 2400 for i in range(4077, 4097)}),  # hubs next to each other, the last ones
    degrees(5000, 20, {i: 2303 + i % 4 for i in range(30)}),  # and the first, around a tile of 2304
    degrees(70000, 10, {i: 3000 for i in range(65530, 65540)}),
    degrees(270000, 1, {7: 6000, 8: 6000, 269999: 4000}),
], ids=["1025", "one", "4097", "5000", "70000", "270000"])
def test_hubs(nemo_mod, oracle_mod, deg):
    n = len(deg)
    rng = np.random.default_rng(n)
    p = Pair(nemo_mod, oracle_mod, rng.uniform(0.0, 0.2, n), rng.uniform(0.0, 2 * np.pi, n), csr=network(deg, n))
    for t in range(2):
        p.step()
    p.check(2)


def test_adjacent_hubs_time(nemo_mod):
    n, count = 20000, 20

    def best(hubs):
        deg = degrees(n, 15, {int(i): 15000 for i in hubs})
        net = nemo_mod.Network()
        rng = np.random.default_rng(2)
        args = np.stack([rng.uniform(0.0, 0.2, n), rng.uniform(0.0, 6.28, n)], axis=1).astype(np.float32)
        net.add_neurons(net.add_neuron_type("Kuramoto"), np.arange(n, dtype=np.uint32), args)
        net.add_synapses_csr(*network(deg, 5))
        sim = nemo_mod.Simulation(net, nemo_mod.Configuration())
        sim.run(5)
        times = []
        for _ in range(5):
            t = time.perf_counter()
            sim.run(5)
            times.append(time.perf_counter() - t)
        return min(times)

    adjacent, spread = best(range(count)), best(np.arange(count) * (n // count))
    assert adjacent < 2.0 * spread, (adjacent, spread)
