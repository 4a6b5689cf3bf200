"""nemo_step by the cycle kernel (csrc/device/cycle_kernel.hip) between runs of
the fused kernel, which share the ring of pending current in memory: every
cycle against the oracle. Sizes at the edges of its workgroups (64 neurons up
to 65536 in all, 256 beyond), one and more than 320 partitions, delays up to
the ring's depth, rows of several chunks of 256 records, buckets with and
without the delay-1 count, every built-in model, stimulus up to 64 entries of
each kind (the kernel's arguments) and beyond (the fused kernel), and dense
firing (left to the fused kernel)."""
import numpy as np
import pytest

from parity import compare_run, same_float

pytestmark = pytest.mark.gpu


def network(n, m, delays, mixed, seed):
    rng = np.random.default_rng(seed)
    k = n - n // 4 if mixed else n
    iz = np.tile(np.array([0.02, 0.2, -65.0, 8.0, 5.0, -13.0, -65.0], np.float32), (k, 1))
    iz[:, 3] -= 6.0 * rng.random(k, dtype=np.float32)
    at = np.arange(n, dtype=np.uint32)
    groups = [("Izhikevich", at[:k], iz)]
    if mixed:
        j = k + n // 8
        ifn = np.tile(np.array([-65.0, -65.0, 1.0, 20.0, 2.0, 5.0, 5.0, -50.0, 0.0, 3.0,
                                -65.0, 0.0, 0.0, 1000.0], np.float32), (j - k, 1))
        groups += [("IF_curr_exp_noise", at[k:j], ifn), ("PoissonSource", at[j:], np.full((n - j, 1), 0.02, np.float32))]
    tgt = rng.integers(0, n, n * m).astype(np.uint32)
    dly = rng.choice(np.array(delays, np.uint8), n * m)
    w = rng.uniform(-0.5, 1.0, n * m).astype(np.float32)
    return groups, np.arange(n + 1, dtype=np.uint64) * m, tgt, dly, w


@pytest.mark.parametrize("n,m,delays,mixed,T", [
    (40, 30, (1,), False, 0),                     # one partition, a ring of two slots
    (1000, 100, tuple(range(1, 21)), False, 0),
    (1000, 700, (1, 2, 63, 64), True, 0),         # rows of three chunks, the deepest ring
    (3001, 40, (1,), True, 512),                  # every record of delay 1: no delay-1 counts
    (25000, 30, (1, 7, 20), False, 64),           # 391 partitions
    (65536, 20, (1, 5, 20), False, 0),
    (65537, 20, (1, 5, 20), True, 0),
])
def test_steps_between_runs(nemo_mod, oracle_mod, n, m, delays, mixed, T):
    groups, rowptr, tgt, dly, w = network(n, m, delays, mixed, n)
    net, orc = nemo_mod.Network(), oracle_mod.Oracle()
    for name, idx, args in groups:
        net.add_neurons(net.add_neuron_type(name), idx, args)
        orc.add_neurons(name, idx, args)
    net.add_synapses_csr(rowptr, tgt, dly, w)
    orc.add_synapses_csr(rowptr, tgt, dly, w)
    orc.finalize()
    conf = nemo_mod.Configuration()
    if T:
        conf.set_partition_size(T)
    sim = nemo_mod.Simulation(net, conf)
    assert sim.info()["fused"] == 1 and sim.info()["saturating"] == 0
    rng = np.random.default_rng(n + 1)
    for run in (3, 40, 1):
        for nf, ni in ((0, 0), (5, 0), (64, 64), (0, 3), (65, 1), (2, 65), (0, 0)):
            fs = rng.integers(0, n, nf).tolist()
            cur = list(zip(rng.integers(0, n, ni).tolist(), rng.uniform(0.0, 40.0, ni).tolist()))
            assert sim.step(fs, cur) == orc.step(fs, cur), (run, nf, ni)
            assert sim.last_kernel_ms() > 0.0
        compare_run(sim, orc, run)
    # a cycle in which every neuron fires, and the dense steps after it
    fs = list(range(n))
    assert sim.step(fs) == orc.step(fs)
    for _ in range(3):
        assert sim.step() == orc.step()
    some = rng.integers(0, n - n // 4, 100)
    for var in range(2):
        got = np.array([sim.get_neuron_state(int(i), var) for i in some], np.float32)
        assert same_float(got, orc.state_all(var)[some])
    counts, ids = sim.read_fired()
    assert len(counts) == 1 and counts[0] == len(ids)
