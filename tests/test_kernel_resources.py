"""What the compiler reports of kernels that hold whole rows in registers:
none may keep part of a row in scratch memory instead."""

import os
import re
import subprocess

import pytest

from fusioninfer_amd.ops.build import CSRC, compile_command


@pytest.mark.parametrize("source", ["norm.hip"])
def test_no_kernel_spills(source):
    hipcc, command = compile_command("_C")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    r = subprocess.run(
        command + ["--cuda-device-only", "-c", os.path.join(CSRC, source),
                   "-o", os.devnull,
                   "-Rpass-analysis=kernel-resource-usage"],
        capture_output=True, text=True, check=True)
    spills = [int(n) for n in re.findall(r"VGPRs Spill: (\d+)", r.stderr)]
    scratch = [int(n) for n in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)",
                                          r.stderr)]
    assert spills and len(spills) == len(scratch)
    assert not any(spills) and not any(scratch)
