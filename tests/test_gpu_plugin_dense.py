"""The plugin step with dense firing, against the oracle: volleys of all
neurons and of a third of them in every cycle, with rows of no, one
and several chunks of 256 synapses and a row longer than all others, at network
sizes of less than a workgroup's 8 neurons, at the edges of 64, and beyond 8
and 64 neurons for each workgroup; without STDP and with it."""
import numpy as np
import pytest

from backends import first_divergence
from parity import compare_run, compare_state, compare_weights
from nemosim_amd import examples

pytestmark = pytest.mark.gpu


def network(n, rows, stdp):
    rng = np.random.default_rng(n)
    args = np.tile(np.array([-65.0, -65.0, 1.0, 20.0, 2.0, 5.0, 5.0, -50.0, 0.0, 3.0,
                             -65.0, 0.0, 0.0, 1000.0], np.float32), (n, 1))
    args[:, 9] += rng.random(n, dtype=np.float32)
    length = rng.choice(np.array(rows), n)
    length[n // 2] = max(rows) * 4
    rowptr = np.zeros(n + 1, np.uint64)
    rowptr[1:] = np.cumsum(length)
    count = int(rowptr[-1])
    w = rng.uniform(-0.5, 0.5, count).astype(np.float32)
    return examples.NetSpec([(examples.IF_CURR_EXP_NOISE, np.arange(n, dtype=np.uint32), args)], rowptr,
                            rng.integers(0, n, count).astype(np.uint32), rng.integers(1, 16, count).astype(np.uint8),
                            w, ((w > 0.0) & bool(stdp)).astype(np.uint8))


@pytest.mark.parametrize("n,rows,learns", [
    (5, (0, 3), False),
    (64, (0, 100, 256, 257), False),
    (65, (1, 1024, 1025), True),
    (2049, (0, 300, 700), True),
    (17001, (20, 60), False),        # more than 8 neurons for each of 2048 workgroups
    (140000, (3, 7), True),          # more than 64 for each
    (270001, (2, 5), True),          # STDP's targets in pieces of 8
])
def test_plugin_step_dense(nemo_mod, oracle_mod, n, rows, learns):
    stdp = examples.stdp_window() + (0.0, 1.0, 0.0, -1.0) if learns else None
    spec = network(n, rows, learns)
    conf = nemo_mod.Configuration()
    conf.set_step_mode("plugins")
    if learns:
        conf.set_stdp_function(stdp[0], stdp[1], min_e=0.0, max_e=1.0, min_i=0.0, max_i=-1.0)
    sim = nemo_mod.Simulation(spec.to_nemo(nemo_mod), conf)
    orc = oracle_mod.from_spec(spec, stdp=stdp)
    assert sim.info()["fused"] == 0
    for k in (40, 1, 2):
        compare_run(sim, orc, k)
        if learns:
            sim.apply_stdp(1.0)
            orc.apply_stdp(1.0)
    fs = [list(range(n)), []] + [list(range(j % 3, n, 3)) for j in range(10)]
    sim.run(len(fs), fstim=fs)
    gc, gi = sim.read_fired()
    ref = [orc.step(f) for f in fs]
    d = first_divergence(np.array([len(f) for f in ref], np.uint32),
                         np.array([i for f in ref for i in f], np.uint32), gc, gi)
    assert d is None, "first diverging cycle %d: %s" % d
    compare_run(sim, orc, 30)
    # synapses delivered: those of every spike
    length = np.diff(spec.rowptr.astype(np.int64))
    assert sim.run(5) == int(length[orc.run(5)[1]].sum())
    compare_state(sim, orc, n, 4, sample=range(0, n, max(1, n // 60)))
    if learns:
        sim.apply_stdp(-0.5)
        orc.apply_stdp(-0.5)
        compare_weights(sim, orc, spec, 2000)
