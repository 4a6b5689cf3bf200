"""STDP on the waves of its own in csrc/device/mask_kernel.hip, against the
oracle (rasters, state, weights bit-exact): a window of one cycle after the
spike and one that fills the 64-cycle history with the delays, rows shorter
and longer than a chunk of 64 synapses, more fired neurons in a wave's words
than it lists at once, more chunks than a work list holds (512), more words
than a wave polls at once, saturating sums, all models, workgroups of more
than 512 neurons, stimuli of more entries than threads, launches of one and
two cycles with rewards between them, and batches."""
import numpy as np
import pytest

from backends import first_divergence
from parity import compare_run, compare_state, compare_weights, hip_sim
from nemosim_amd import examples

pytestmark = pytest.mark.gpu


def window(length_pre, length_post):
    pre, post = examples.stdp_window(length=64)
    return list(pre[:length_pre]), list(post[:length_post])


@pytest.mark.parametrize("kind,n,m,dmax,T,pre,post,max_e", [
    ("iz", 1000, 100, 20, 0, 20, 20, 1.0),
    ("iz", 1000, 100, 20, 64, 30, 1, 1.0),        # the shortest window after the spike
    ("iz", 1500, 200, 44, 192, 20, 20, 1.0),      # delays and window fill the history
    ("iz", 2000, 700, 1, 128, 10, 5, 1.0),        # delay 1 only, rows of several chunks
    ("iz", 5000, 5, 3, 320, 20, 20, 1.0),         # rows of a few synapses
    ("iz", 20000, 20, 9, 64, 20, 20, 1.0),        # 626 words for a workgroup's one wave
    ("if", 1500, 300, 20, 256, 20, 20, 1.0),      # a third of the neurons fires each cycle
    ("iz", 1200, 150, 20, 128, 20, 20, 1500.0),   # saturating
    ("if", 1200, 150, 20, 448, 20, 20, 1500.0),
    ("iz", 140000, 4, 5, 0, 20, 20, 1.0),         # 576 neurons, 6 waves for STDP
])
def test_mask_stdp(nemo_mod, oracle_mod, kind, n, m, dmax, T, pre, post, max_e):
    make = examples.izhikevich_80_20 if kind == "iz" else examples.if_curr_exp_80_20
    spec = make(n, m, seed=n + T, dmax=dmax, stdp=True)
    stdp = window(pre, post) + (0.0, max_e, 0.0, -max_e)
    sim = hip_sim(nemo_mod, spec, stdp=stdp, partition_size=T or None)
    orc = oracle_mod.from_spec(spec, stdp=stdp)
    info = sim.info()
    assert info["block_threads"] > info["partition_size"], info   # waves for STDP
    assert info["saturating"] == (1 if max_e > 1.0 else 0), info
    long = n < 100000
    for k in (60, 1, 2) + ((40, 1, 25) if long else (2,)):
        compare_run(sim, orc, k)
        sim.apply_stdp(0.5)
        orc.apply_stdp(0.5)
    rng = np.random.default_rng(n)
    # a burst of every neuron, then stimuli of more entries than threads
    fs = [list(range(n)) if j == 1 else rng.integers(0, n, 1100 if j % 4 == 0 else 3).tolist()
          for j in range(post + 12)]
    sim.run(len(fs), fstim=fs)
    gc, gi = sim.read_fired()
    ref = [orc.step(f) for f in fs]
    d = first_divergence(np.array([len(f) for f in ref], np.uint32),
                         np.array([i for f in ref for i in f], np.uint32), gc, gi)
    assert d is None, "first diverging cycle %d: %s" % d
    sim.apply_stdp(-0.5)
    orc.apply_stdp(-0.5)
    compare_run(sim, orc, 30 if long else 3)
    compare_state(sim, orc, spec.n, 2, sample=range(0, spec.n, max(1, n // 60)))
    compare_weights(sim, orc, spec, 2000, seed=3)


def test_mask_stdp_batch(nemo_mod, oracle_mod):
    """networks of different workgroup sizes in one launch, alternating with
    launches of their own"""
    stdp = window(20, 20) + (0.0, 1.0, 0.0, -1.0)
    specs = [examples.izhikevich_80_20(n, 80, seed=n, stdp=True) for n in (300, 3000, 7000)]
    sims = [hip_sim(nemo_mod, s, stdp=stdp) for s in specs]
    orcs = [oracle_mod.from_spec(s, stdp=stdp) for s in specs]
    assert len({s.info()["block_threads"] for s in sims}) > 1
    for steps, batched in [([40, 90, 1], True), ([3, 1, 20], False), ([25, 2, 60], True)]:
        if batched:
            nemo_mod.run_batch(sims, steps)
        for sim, orc, k in zip(sims, orcs, steps):
            if batched:
                gc, gi = sim.read_fired()
                rc, ri = orc.run(k)
                d = first_divergence(rc, ri, gc, gi)
                assert d is None, "first diverging cycle %d: %s" % d
            else:
                compare_run(sim, orc, k)
            sim.apply_stdp(1.0)
            orc.apply_stdp(1.0)
    for sim, orc, s in zip(sims, orcs, specs):
        compare_weights(sim, orc, s, 1500, seed=1)
