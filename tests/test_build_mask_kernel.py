"""Properties of the build (CPU): every variant of the word-exchanging step
kernel (csrc/device/mask_kernel.hip), for one network and for batches, fits the
128 VGPRs a 1024-thread workgroup allows without spilling to scratch memory."""
import os
import re

import pytest

from test_build import kernel_resources

REPORT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "nemosim_amd", "_build",
                      "mask_kernel.resources.txt")


def report():
    if not os.path.exists(REPORT):
        pytest.skip("no build report (build with __graft_entry__.build())")
    with open(REPORT) as f:
        return f.read()


def test_mask_kernels_do_not_spill():
    res = {k: v for k, v in kernel_resources(report()).items() if "nemo_mask_kernel" in k}
    assert len(res) == 22, sorted(res)
    for name, (vgprs, scratch) in res.items():
        assert vgprs is not None and vgprs <= 128, (name, vgprs)
        assert scratch == 0, "%s spills %d bytes per lane" % (name, scratch)
