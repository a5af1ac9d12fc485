"""The device FEM's solve for many bodies leaves room for a second one on its CU: at
most 256 registers a lane (two wavefronts a SIMD) and none of them kept in memory,
as the compiler reports it."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "life_amd", "csrc")


def test_two_bodies_a_cu():
    flags = subprocess.run(["make", "-s", "-C", CSRC, "--eval", "flags: ; @echo $(HIPCC) $(HIPFLAGS)", "flags"],
                           check=True, capture_output=True, text=True).stdout.split()
    if not shutil.which(flags[0]):
        pytest.skip("no compiler for the device")
    out = subprocess.run(flags + ["-ffp-contract=off", "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage",
                                  "-c", "fem_dev.hip", "-o", os.devnull], cwd=CSRC, check=True, capture_output=True,
                         text=True).stderr
    kernels = {}
    for line in out.splitlines():
        m = re.search(r"remark:\s+(.+?): (\S+) \[-Rpass", line)
        if m and m.group(1) == "Function Name":
            kernels[m.group(2)] = use = {}
        elif m:
            use[m.group(1)] = int(m.group(2)) if m.group(2).isdigit() else m.group(2)
    found = {k: u for k, u in kernels.items() if "k_fem_dynamicILi256ELb1E" in k}
    assert len(found) == 1
    for name, use in found.items():
        print(name, use)
        assert use["Occupancy [waves/SIMD]"] >= 2
        assert use["ScratchSize [bytes/lane]"] == 0 and use["VGPRs Spill"] == 0
