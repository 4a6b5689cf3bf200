"""Simulations of every kernel variant built, run and stepped by several
threads at once, each against the oracle: what construction asks of the device
(occupancy, LDS limits) is kept in tables that all threads share."""
import threading

import pytest

from parity import compare_run
from nemosim_amd import examples

pytestmark = pytest.mark.gpu


def test_threads(nemo_mod, oracle_mod):
    errors = []

    def work(k):
        try:
            for n in (300 + 70 * k, 5000 + 900 * k):
                stdp = examples.stdp_window() + (0.0, 1.0, 0.0, -1.0) if k & 1 else None
                make = examples.if_curr_exp_80_20 if k & 2 else examples.izhikevich_80_20
                spec = make(n, 40, seed=n, stdp=bool(stdp))
                if k & 4:
                    spec.weights = spec.weights * spec.weights.dtype.type(2000.0)   # sums that leave int32
                conf = nemo_mod.Configuration()
                if stdp:
                    conf.set_stdp_function(stdp[0], stdp[1], min_e=0.0, max_e=1.0, min_i=0.0, max_i=-1.0)
                if k & 8:
                    conf.set_partition_size(64)
                sim = nemo_mod.Simulation(spec.to_nemo(nemo_mod), conf)
                orc = oracle_mod.from_spec(spec, stdp=stdp)
                compare_run(sim, orc, 15)
                assert sim.step([1, 2, 3]) == orc.step([1, 2, 3])
        except BaseException as e:   # noqa: B902 -- reported by the test's thread
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(16)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
