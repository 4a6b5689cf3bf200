"""nemo_set_exchange_waves(conf, -1): no wave is set apart, neither for the
exchange nor for the records of longer delays, whichever way a network
exchanges its spikes; by default the latter have waves of their own. Rasters
against the oracle, alone and in a batch."""
import pytest

from backends import first_divergence
from parity import compare_run
from nemosim_amd import examples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,T", [(1000, 100, 0), (6000, 200, 256), (20000, 60, 512)])
def test_no_waves_apart(nemo_mod, oracle_mod, n, m, T):
    spec = examples.izhikevich_80_20(n, m, seed=n)
    orc = oracle_mod.from_spec(spec)
    sims = []
    for waves in (-1, 0):
        conf = nemo_mod.Configuration()
        conf.set_exchange_waves(waves)
        if T:
            conf.set_partition_size(T)
        sims.append(nemo_mod.Simulation(spec.to_nemo(nemo_mod), conf))
    none, auto = [s.info() for s in sims]
    assert none["exchange_waves"] == 0 and none["far_list_sources"] == 0, none
    assert none["block_threads"] == none["partition_size"], none
    assert auto["block_threads"] > auto["partition_size"], auto
    for k in (1, 50, 120):
        compare_run(sims[0], orc, k)
    nemo_mod.run_batch(sims, [30, 201])
    rc, ri = orc.run(30)
    gc, gi = sims[0].read_fired()
    assert first_divergence(rc, ri, gc, gi) is None
