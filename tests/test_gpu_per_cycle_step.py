"""The per-cycle step of built-in models (csrc/device/plugin_step.hip,
pm_cycle_kernel): networks beyond the fused kernel's range. A count that fills
neither a workgroup of 256 nor a raster word, all built-in models in one
network or Izhikevich alone, sums that stay within int32 or leave it (int64
accumulators), delays up to the ring's whole depth, stimulus in single steps
between runs; every raster and the state against the oracle."""
import numpy as np
import pytest

from parity import compare_run, same_float

pytestmark = pytest.mark.gpu

DMAX = 64


def groups(n, mixed, rng):
    iz = np.tile(np.array([0.02, 0.2, -65.0, 8.0, 5.0, -13.0, -65.0], np.float32), (n, 1))
    iz[:, 3] -= 6.0 * rng.random(n, dtype=np.float32)
    if not mixed:
        return [("Izhikevich", np.arange(n, dtype=np.uint32), iz)]
    k = n - 1000
    ifn = np.tile(np.array([-65.0, -65.0, 1.0, 20.0, 2.0, 5.0, 5.0, -50.0, 0.0, 3.0,
                            -65.0, 0.0, 0.0, 1000.0], np.float32), (600, 1))
    at = np.arange(n, dtype=np.uint32)
    return [("Izhikevich", at[:k], iz[:k]), ("IF_curr_exp_noise", at[k:k + 600], ifn),
            ("PoissonSource", at[k + 600:k + 900], np.full((300, 1), 0.05, np.float32)),
            ("Input", at[k + 900:], np.zeros((100, 0), np.float32))]


@pytest.mark.parametrize("n,mixed,gain", [(90001, True, 1.0), (90047, False, 1.0), (90048, True, 1900.0),
                                          (90113, False, 1900.0)])
def test_per_cycle_step(nemo_mod, oracle_mod, n, mixed, gain):
    rng = np.random.default_rng(n)
    m = 8
    rowptr = np.arange(n + 1, dtype=np.uint64) * m
    tgt = rng.integers(0, n, n * m).astype(np.uint32)
    dly = rng.choice(np.array([1, 2, 3, DMAX - 1, DMAX], np.uint8), n * m)
    w = (rng.uniform(-0.5, 1.0, n * m) * gain).astype(np.float32)
    net, orc = nemo_mod.Network(), oracle_mod.Oracle()
    for name, idx, args in groups(n, mixed, rng):
        net.add_neurons(net.add_neuron_type(name), idx, args)
        orc.add_neurons(name, idx, args)
    net.add_synapses_csr(rowptr, tgt, dly, w)
    orc.add_synapses_csr(rowptr, tgt, dly, w)
    orc.finalize()
    sim = nemo_mod.Simulation(net, nemo_mod.Configuration())
    info = sim.info()
    assert info["fused"] == 0 and info["saturating"] == (1 if gain > 1.0 else 0), info
    compare_run(sim, orc, 70)
    for t in range(6):
        fs = rng.integers(0, n, 300 * (t % 2)).tolist()
        cur = list(zip(rng.integers(0, n, 200).tolist(), rng.uniform(0.0, 30.0, 200).tolist())) if t != 3 else []
        assert sim.step(fs, cur) == orc.step(fs, cur), t
    compare_run(sim, orc, 70)
    some = rng.integers(0, n - 1000, 200)
    for var in range(2):
        got = np.array([sim.get_neuron_state(int(i), var) for i in some], np.float32)
        assert same_float(got, orc.state_all(var)[some])
