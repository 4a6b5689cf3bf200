"""The persistent step that exchanges fired bits as words
(csrc/device/mask_kernel.hip), against the oracle at the edges of its parts:
the words a wave takes (64 and 256, and more than its largest form polls at
once), lists of 128 sources per wave and many lists (every neuron forced to
fire), partitions that are not full, stimulus schedules of one cycle and of
more entries than threads, launches of one, two and three cycles, records of
the longest delay without the delay-1 count, saturating sums, all models."""
import numpy as np
import pytest

from parity import compare_state
from backends import first_divergence

pytestmark = pytest.mark.gpu


def build(nemo_mod, oracle_mod, n, m, delays, mixed=False, gain=1.0, T=0):
    rng = np.random.default_rng(n + m)
    k = n - n // 3 if mixed else n
    iz = np.tile(np.array([0.02, 0.2, -65.0, 8.0, 5.0, -13.0, -65.0], np.float32), (k, 1))
    iz[:, 3] -= 6.0 * rng.random(k, dtype=np.float32)
    at = np.arange(n, dtype=np.uint32)
    groups = [("Izhikevich", at[:k], iz)]
    if mixed:
        ifn = np.tile(np.array([-65.0, -65.0, 1.0, 20.0, 2.0, 5.0, 5.0, -50.0, 0.0, 3.0,
                                -65.0, 0.0, 0.0, 1000.0], np.float32), (n - k, 1))
        groups.append(("IF_curr_exp_noise", at[k:], ifn))
    rowptr = np.arange(n + 1, dtype=np.uint64) * m
    tgt = rng.integers(0, n, n * m).astype(np.uint32)
    dly = rng.choice(np.array(delays, np.uint8), n * m)
    w = (rng.uniform(-0.5, 0.7, n * m) * gain).astype(np.float32)
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
    assert sim.info()["fused"] == 1
    return sim, orc


def check(sim, orc, cycles, fstim=None, istim=None):
    sim.run(cycles, fstim=fstim, istim=istim)
    gc, gi = sim.read_fired()
    ref = [orc.step(fstim[k] if fstim else None, istim[k] if istim else None) for k in range(cycles)]
    rc = np.array([len(f) for f in ref], np.uint32)
    ri = np.array([i for f in ref for i in f], np.uint32)
    d = first_divergence(rc, ri, gc, gi)
    assert d is None, "first diverging cycle %d: %s" % d


@pytest.mark.parametrize("n,m,delays,mixed,gain,T", [
    (2048, 60, tuple(range(1, 21)), False, 1.0, 64),   # 64 words for the partition's one wave
    (2049, 60, tuple(range(1, 21)), False, 1.0, 64),   # 66
    (8192, 30, (1, 2, 20), False, 1.0, 64),            # 256
    (8193, 30, (1, 2, 20), True, 1.0, 64),             # 258
    (20000, 20, (1, 9), False, 1.0, 64),               # 626: more than one poll
    (700, 50, (1,), True, 1.0, 0),                     # every record of delay 1
    (1000, 90, (1, 2, 64), True, 1.0, 192),            # the deepest ring, a partition of 40
    (1500, 200, (1, 5, 20), False, 900.0, 128),        # saturating
    (1300, 200, (3, 20), True, 900.0, 320),
    (513, 600, (1, 2, 3), False, 1.0, 0),              # buckets longer than a pass
    (6000, 40, (1, 2, 20), True, 1.0, 320),            # five waves, more sources than the far list holds (1280)
    (6000, 40, (1, 2, 20), True, 1.0, 640),            # ten waves and six for far records
])
def test_mask_kernel(nemo_mod, oracle_mod, n, m, delays, mixed, gain, T):
    sim, orc = build(nemo_mod, oracle_mod, n, m, delays, mixed, gain, T)
    assert sim.info()["saturating"] == (1 if gain > 1.0 else 0)
    rng = np.random.default_rng(n)

    def stim(k, nf, ni):
        f = [rng.integers(0, n, nf if j % 3 else 0).tolist() for j in range(k)]
        i = [list(zip(rng.integers(0, n, ni).tolist(), rng.uniform(0.0, 40.0, ni).tolist())) if j % 2 else []
             for j in range(k)]
        return f, i

    check(sim, orc, 40)
    for k in (1, 2, 3, 7):
        check(sim, orc, k, *stim(k, 5, 4))
    check(sim, orc, 6, *stim(6, 1200, 1100))           # more entries than threads
    check(sim, orc, 5, fstim=[list(range(n))] * 3 + [[]] * 2)   # several lists per wave
    check(sim, orc, 30)
    if gain == 1.0:
        compare_state(sim, orc, n, 2, sample=range(0, n - n // 3, 29))


def test_mask_kernel_batch(nemo_mod, oracle_mod):
    """partitions of different sizes in one launch: waves beyond a network's
    own partition size only keep the barriers"""
    pairs = [build(nemo_mod, oracle_mod, n, 60, (1, 2, 20), T=T)
             for n, T in ((900, 64), (3000, 512), (2500, 192), (64, 64), (5000, 960))]
    for steps in ([50] * 5, [3, 70, 1, 20, 33]):
        nemo_mod.run_batch([s for s, _ in pairs], steps)
        for (sim, orc), k in zip(pairs, steps):
            rc, ri = orc.run(k)
            gc, gi = sim.read_fired()
            assert first_divergence(rc, ri, gc, gi) is None
