"""Batched launches of the step that exchanges words, where the networks differ
from the common ones: sums that leave int32, without STDP and with it; one or
all models; a member of more partitions than a wave polls words of at once
(256); packs whose members all fit with far waves and packs that do not; in
turn with launches of their own. Rasters, state and weights against the
oracle."""
import numpy as np
import pytest

from backends import first_divergence
from parity import compare_run, compare_state, compare_weights, hip_sim
from test_gpu_mask_kernel import build
from nemosim_amd import examples

pytestmark = pytest.mark.gpu


def in_turn(nemo_mod, pairs, rounds, after=None):
    """batched and own launches in turn, every raster against the oracle"""
    rng = np.random.default_rng(len(pairs))
    for r in range(rounds):
        steps = [int(k) for k in rng.integers(1, 40, len(pairs))]
        if r % 3 != 2:
            nemo_mod.run_batch([s for s, _ in pairs], steps)
        for (sim, orc), k in zip(pairs, steps):
            if r % 3 == 2:
                compare_run(sim, orc, k)
            else:
                gc, gi = sim.read_fired()
                rc, ri = orc.run(k)
                d = first_divergence(rc, ri, gc, gi)
                assert d is None, "round %d: first diverging cycle %d: %s" % ((r,) + d)
            if after:
                after(sim, orc)


@pytest.mark.parametrize("mixed", [False, True])
def test_saturating(nemo_mod, oracle_mod, mixed):
    sizes = ((700, 64), (2500, 192), (1500, 320), (300, 0), (3000, 512))
    pairs = [build(nemo_mod, oracle_mod, n, 150, (1, 2, 20), mixed=mixed, gain=900.0, T=T) for n, T in sizes]
    assert all(s.info()["saturating"] == 1 for s, _ in pairs)
    in_turn(nemo_mod, pairs, 6)
    for (sim, orc), (n, _) in zip(pairs, sizes):
        compare_state(sim, orc, n, 2, sample=range(0, n - n // 3, 41))


@pytest.mark.parametrize("kind", ["iz", "if"])
def test_saturating_stdp(nemo_mod, oracle_mod, kind):
    stdp = examples.stdp_window() + (0.0, 1500.0, 0.0, -1500.0)
    make = examples.izhikevich_80_20 if kind == "iz" else examples.if_curr_exp_80_20
    sizes = ((400, 64), (1500, 128), (2600, 256))
    specs = [make(n, 150, seed=n, stdp=True) for n, _ in sizes]
    pairs = [(hip_sim(nemo_mod, s, stdp=stdp, partition_size=T), oracle_mod.from_spec(s, stdp=stdp))
             for s, (_, T) in zip(specs, sizes)]
    assert all(s.info()["saturating"] == 1 for s, _ in pairs)

    def reward(sim, orc):
        sim.apply_stdp(0.5)
        orc.apply_stdp(0.5)

    in_turn(nemo_mod, pairs, 6, reward)
    for (sim, orc), spec in zip(pairs, specs):
        compare_state(sim, orc, spec.n, 2, sample=range(0, spec.n, 37))
        compare_weights(sim, orc, spec, 1500, seed=2)


@pytest.mark.parametrize("gain", [1.0, 900.0])
def test_many_partitions(nemo_mod, oracle_mod, gain):
    """9000 neurons in 141 partitions of 64: 282 words for each one's wave"""
    m = 30 if gain == 1.0 else 150
    pairs = [build(nemo_mod, oracle_mod, n, m, (1, 2, 20), gain=gain, T=T) for n, T in ((9000, 64), (1200, 64), (2000, 256))]
    assert pairs[0][0].info()["partitions"] == 141
    in_turn(nemo_mod, pairs, 5)


def test_pack_that_far_waves_do_not_fit(nemo_mod, oracle_mod):
    """about as many workgroups as the device holds: no room for far waves,
    which the same members have in a pack of their own"""
    pairs = [build(nemo_mod, oracle_mod, 4000 + 64 * i, 20, (1, 2, 20), T=64) for i in range(24)]
    in_turn(nemo_mod, pairs, 2)
    in_turn(nemo_mod, pairs[:3], 4)
