"""nemo_step and batched runs of the same simulations in turn, against the
oracle. A step's kernel reports to the host from within, a batched launch has
a stream of its own: it is ordered after the end of every member's last step,
so that it finds the step's state, ring and history. Members that were stepped,
that ran alone (whose report resets the launch clock that the batch uses too)
and that did neither are in one batch."""
import numpy as np
import pytest

from backends import first_divergence
from parity import compare_run, compare_state, hip_sim
from nemosim_amd import examples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,m", [((64, 1000, 3000), 100), ((20000, 70000), 60)])
def test_steps_and_batches_in_turn(nemo_mod, oracle_mod, sizes, m):
    specs = [examples.izhikevich_80_20(n, m, seed=n + 7) for n in sizes]
    sims = [hip_sim(nemo_mod, s) for s in specs]
    orcs = [oracle_mod.from_spec(s) for s in specs]
    rng = np.random.default_rng(len(sizes))
    for turn in range(25):
        for k, (sim, orc, spec) in enumerate(zip(sims, orcs, specs)):
            if (turn + k) % 3 == 0:
                compare_run(sim, orc, 2)
            elif (turn + k) % 3 == 1:
                fs = rng.integers(0, spec.n, 8).tolist()
                assert sim.step(fs) == orc.step(fs), (turn, spec.n)
        last = len(sims) - 1
        assert sims[last].step() == orcs[last].step(), turn     # the call right before the batch
        steps = [int(k) for k in rng.integers(1, 5, len(sims))]
        nemo_mod.run_batch(sims, steps)
        for sim, orc, k in zip(sims, orcs, steps):
            assert 0.0 < sim.last_kernel_ms() < 1000.0, turn
            gc, gi = sim.read_fired()
            rc, ri = orc.run(k)
            d = first_divergence(rc, ri, gc, gi)
            assert d is None, "turn %d: first diverging cycle %d: %s" % ((turn,) + d)
    for sim, orc, spec in zip(sims, orcs, specs):
        compare_state(sim, orc, spec.n, 2, sample=range(0, spec.n, max(1, spec.n // 50)))
