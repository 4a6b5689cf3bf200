"""nemo_hip_read_fired counts and lists the spikes of a run on the device
(csrc/device/raster_kernel.hip). Checked against the raw raster decoded here,
at one cycle, at the edges of its passes (16384 neurons), of its windows of 2^18
ids and of its groups of 16384 cycles, in one call and in two (from 2^22 bits),
with contiguous and scattered user indices."""
import ctypes

import numpy as np
import pytest

import nemosim_amd
from nemosim_amd import _lib

pytestmark = pytest.mark.gpu


def forced_network(idx):
    """Input neurons: they fire exactly when forced"""
    net = nemosim_amd.Network()
    t = net.add_neuron_type("Input")
    net.add_neurons(t, idx, np.zeros((len(idx), 0), np.float32))
    return nemosim_amd.Simulation(net, nemosim_amd.Configuration())


def decoded(sim, idx):
    raster = sim.read_raster()
    bits = np.unpackbits(raster.view(np.uint8), axis=1, bitorder="little")[:, :len(idx)]
    return bits.sum(axis=1).astype(np.uint32), np.concatenate([idx[np.flatnonzero(b)] for b in bits])


@pytest.mark.parametrize("n,first,step,cycles,rate", [
    (63, 5, 1, 4, 0.5),
    (64, 2, 1, 1, 0.5),
    (64, 0, 3, 12288, 0.02),
    (65, 0, 3, 6145, 0.02),       # two words
    (16384, 0, 1, 49, 0.01),      # one pass per cycle
    (16385, 7, 1, 60, 1.0),       # one id past a pass; 655k ids: three windows
    (20001, 3, 2, 50, 1.0),       # scattered ids over three windows
    (70, 0, 1, 16390, 0.02),      # two groups of cycles
    (64, 0, 3, 65536, 0.05),      # the most that one call reads, in four groups
    (65, 0, 3, 32769, 0.05),      # two calls
])
def test_read_fired_equals_raster(n, first, step, cycles, rate):
    rng = np.random.default_rng(n)
    idx = (first + step * np.arange(n)).astype(np.uint32)
    sim = forced_network(idx)
    stim = [idx[rng.random(n) < rate] if k % 3 else idx[:0] for k in range(cycles)]
    sim.run(cycles, fstim=stim)
    counts, ids = sim.read_fired()
    rc, ri = decoded(sim, idx)
    assert np.array_equal(counts, [len(s) for s in stim])
    assert np.array_equal(counts, rc)
    assert np.array_equal(ids, ri)


@pytest.mark.parametrize("quiet", [0, 6200])
def test_read_fired_small_buffer(quiet):
    """a buffer that ends inside a cycle receives the cycles before it (with
    6200 quiet cycles after them, too)"""
    idx = np.arange(100, dtype=np.uint32)
    sim = forced_network(idx)
    sim.run(3 + quiet, fstim=[idx[:10], idx[20:50], idx] + [[]] * quiet)
    lib = _lib.load()
    counts = np.full(3 + quiet, 77, np.uint32)
    ids = np.full(60, 999, np.uint32)
    total = ctypes.c_size_t()
    st = lib.nemo_hip_read_fired(sim._h, counts.ctypes.data_as(_lib.c_uint_p), ids.ctypes.data_as(_lib.c_uint_p), 60,
                                 ctypes.byref(total))
    assert st != 0
    assert list(counts[:3]) == [10, 30, 100]
    assert (counts[3:] == 77).all()
    assert list(ids[:40]) == list(range(10)) + list(range(20, 50))
    assert (ids[40:] == 999).all()
