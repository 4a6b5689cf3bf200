"""Flags of the build (CPU): every compilation for the device asks for IEEE
square roots and divisions and leaves out contraction and packed FP32, on which
bit parity of the neuron models rests; nothing asks for fast math."""
import os
import subprocess

DIR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "nemosim_amd")


def test_device_flags():
    out = subprocess.run(["make", "-n", "-B", "-C", DIR], check=True, capture_output=True, text=True).stdout
    lines = [l for l in out.replace("\\\n", " ").splitlines() if "--offload-arch" in l and ".hip" in l]
    assert len(lines) >= 12, out
    for line in lines:
        for flag in ("-fhip-fp32-correctly-rounded-divide-sqrt", "-ffp-contract=off", "-packed-fp32-ops"):
            assert flag in line, (flag, line)
        assert "fast-math" not in line
