"""device_bytes of nemo_hip_get_info holds what the exchange between partitions
takes: two networks that differ in the number of partitions only differ by
their rings' padding, the bucket bounds and, for words, 8 bytes for each 32
neurons and kept cycle (lines of 128), with STDP postLen + 3 cycles."""
import pytest

from parity import hip_sim
from nemosim_amd import examples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stdp_on", [False, True])
def test_exchange_words_counted(nemo_mod, stdp_on):
    n, m = 4096, 50
    stdp = examples.stdp_window() + (0.0, 1.0, 0.0, -1.0) if stdp_on else None
    spec = examples.izhikevich_80_20(n, m, seed=1, stdp=stdp_on)
    sim = hip_sim(nemo_mod, spec, stdp=stdp, partition_size=128)
    info = sim.info()
    p, t, d = info["partitions"], info["partition_size"], info["max_delay"]
    assert (p, t, info["fused"], info["exchange_waves"]) == (32, 128, 1, 0)
    neuron = 1 + 10 * 4 + 4 * 4 + 16 + 8              # model, parameters, state, RNG, history
    expect = n * neuron + p * 2 * (d + 1) * t * 4 + (n * (p + 1) + 1) * 4 + n * m * 8
    kept = 20 + 3 if stdp_on else 2
    expect += kept * (p * t // 32) * 8
    if stdp_on:
        plastic = info["plastic_synapses"]
        expect += 4 * n * 8 + (n + 1) * 4 + plastic * 12    # histories, reverse matrix and accumulators
    assert info["device_bytes"] == expect
