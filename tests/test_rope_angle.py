"""The decode step forms its rotary table entries without a branch, by its own fp64
sine and cosine.  This CPU test builds that function for the host and compares
it, bit for bit in fp32, with the host library's (the oracle's formula): every
position of the contexts the engine is configured for, and strided ones up to
2^31."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_rope_entries_match_the_host_library(tmp_path):
    exe = tmp_path / "rope_angle_check"
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-mfma", "-ffp-contract=off", "-std=c++17", "-x", "hip",
                    os.path.join(HERE, "csrc", "rope_angle_check.cpp"), "-o", str(exe)], check=True, capture_output=True)
    for first, end, step in ((0, 262144, 1), (262144, 1 << 24, 37), (1 << 24, (1 << 31) - 20000, 10007)):
        n, bad = map(int, subprocess.run([str(exe), str(first), str(end), str(step)], check=True, capture_output=True,
                                         text=True).stdout.split())
        assert n >= 32 * 200000 and bad == 0, (first, end, n, bad)
