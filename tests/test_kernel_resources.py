"""Registers of the warm start's ring convolutions, from the compiler's own
report: none of them spills (16 -> 48 channels at rows of 32 positions did when
the gate of the backward direction was a run-time choice)."""
import os
import re
import subprocess

import pytest

from physis_amd import build


def test_ring_convolutions_do_not_spill(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("hipcc not available")
    p = subprocess.run(
        [build.HIPCC, *build.HIP_FLAGS, "--cuda-device-only", "-S",
         "-Rpass-analysis=kernel-resource-usage", build.WARMSTART_SOURCES[0],
         "-o", str(tmp_path / "unet.s")], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-2000:]
    name, spilled = "", {}
    for line in p.stderr.splitlines():
        m = re.search(r"remark:.* Name: (\S+)", line)
        if m:
            name = m.group(1)
        m = re.search(r"VGPRs Spill: (\d+)", line)
        if m and "ConvZKernel" in name:
            spilled[name] = int(m.group(1))
    assert len(spilled) >= 20  # the widths of the seven layers, by direction
    assert not any(spilled.values()), {k: v for k, v in spilled.items() if v}
