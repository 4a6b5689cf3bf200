"""nemo_step's one-cycle kernel keeps a source's bucket bounds, one for each
partition and wave, in LDS (CPU). A configured partition of 64 neurons gives a
network of a quarter of a million about 4000 partitions, whose bounds do not
fit: the host has to know, since the launch would fail, and take the fused
kernel."""
import pytest

from nemosim_amd import _lib

STATIC = 2 * 256 * 4 + 8 * 4 + 2 * 4 * 4 + 4 * 8      # the kernel's own variables


@pytest.mark.parametrize("partitions", [1, 391, 1563, 3839, 3840, 3960, 4096, 1 << 20, (1 << 32) - 1])
def test_bounds_fit_the_launch(partitions):
    fits = _lib.load().nemo_dev_cycle_fits
    fits.argtypes = [_lib.ctypes.c_uint32]
    total = 4 * (partitions + 1) * 4 + STATIC
    if fits(partitions):
        assert total <= 64 * 1024
    else:
        assert partitions > 3000                       # and no network is turned away early
