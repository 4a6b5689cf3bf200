"""The per-cycle step of networks with long rows next to each other
(pm_cycle_kernel without its delivery, then pm_scatter_kernel): 16 and more
neighbours whose synapses are more than a workgroup should deliver, beside
neurons with few and with none, with int32 and int64 accumulators, all
built-in models and STDP, forced and in volleys of all neurons, against the
oracle."""
import numpy as np
import pytest

from backends import first_divergence
from parity import compare_run, compare_state, compare_weights
from nemosim_amd import examples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,first,hubs,row,gain,dmax,stdp_on", [
    (90001, 0, 20, 1200, 1.0, 64, False),
    (90047, 90047 - 17, 17, 1500, 900.0, 64, False),     # the last neurons; sums that leave int32
    (140048, 160, 16, 1100, 1.0, 44, True),               # one piece of 16
])
def test_long_rows(nemo_mod, oracle_mod, n, first, hubs, row, gain, dmax, stdp_on):
    rng = np.random.default_rng(n)
    args = np.tile(np.array([0.02, 0.2, -65.0, 8.0, 5.0, -13.0, -65.0], np.float32), (n, 1))
    length = rng.integers(0, 8, n)
    length[first:first + hubs] = row
    rowptr = np.zeros(n + 1, np.uint64)
    rowptr[1:] = np.cumsum(length)
    count = int(rowptr[-1])
    w = (rng.uniform(-0.5, 1.0, count) * gain).astype(np.float32)
    # a thousand targets take a third of the synapses, so that sums grow
    tgt = np.where(rng.random(count) < 0.3, rng.integers(0, 1000, count), rng.integers(0, n, count)).astype(np.uint32)
    spec = examples.NetSpec([(examples.IZHIKEVICH, np.arange(n, dtype=np.uint32), args)], rowptr, tgt,
                            rng.choice(np.array([1, 2, 3, dmax - 1, dmax], np.uint8), count), w,
                            ((w > 0.0) & stdp_on).astype(np.uint8))
    stdp = examples.stdp_window() + (0.0, 1.0, 0.0, -1.0) if stdp_on else None
    conf = nemo_mod.Configuration()
    if stdp:
        conf.set_stdp_function(stdp[0], stdp[1], min_e=0.0, max_e=1.0, min_i=0.0, max_i=-1.0)
    sim = nemo_mod.Simulation(spec.to_nemo(nemo_mod), conf)
    info = sim.info()
    assert info["fused"] == 0 and info["saturating"] == (1 if gain > 1.0 else 0), info
    orc = oracle_mod.from_spec(spec, stdp=stdp)
    some = list(range(first, first + hubs))
    compare_run(sim, orc, 20)
    assert sim.step(some) == orc.step(some)
    fs = [some, [], list(range(n)), some[::2]] + [[]] * 46
    events = sim.run(len(fs), fstim=fs)
    gc, gi = sim.read_fired()
    ref = [orc.step(f) for f in fs]
    ids = np.array([i for f in ref for i in f], np.uint32)
    d = first_divergence(np.array([len(f) for f in ref], np.uint32), ids, gc, gi)
    assert d is None, "first diverging cycle %d: %s" % d
    assert events == int(length[ids].sum())
    if stdp:
        sim.apply_stdp(1.0)
        orc.apply_stdp(1.0)
    compare_run(sim, orc, 20)
    compare_state(sim, orc, n, 2, sample=some + list(range(0, n, n // 60)))
    if stdp:
        compare_weights(sim, orc, spec, 2000)
