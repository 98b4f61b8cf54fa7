"""What the compiler reports of kernels that hold whole rows in registers:
none may keep part of a row in scratch memory instead."""

import os
import re
import subprocess

import pytest

from fusioninfer_amd.ops.build import CSRC, compile_command


@pytest.mark.parametrize("source,kernels", [
    ("norm.hip", ""),
    # reads of scratch memory wait for the stores and copies in front of them
    ("prefill_attention.hip", "prefill_(rows|attn)_kernel"),
    ("seqmix_sink.hip", "prefill_rows_kernel"),
])
def test_no_kernel_spills(source, kernels):
    hipcc, command = compile_command("_C")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    r = subprocess.run(
        command + ["--cuda-device-only", "-c", os.path.join(CSRC, source),
                   "-o", os.devnull,
                   "-Rpass-analysis=kernel-resource-usage"],
        capture_output=True, text=True, check=True)
    names = re.findall(r"Function Name: (\S+)", r.stderr)
    spills = [int(n) for n in re.findall(r"VGPRs Spill: (\d+)", r.stderr)]
    scratch = [int(n) for n in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)",
                                          r.stderr)]
    assert len(names) == len(spills) == len(scratch)
    found = [n for n in zip(names, spills, scratch) if re.search(kernels, n[0])]
    assert found and not [n for n in found if n[1] or n[2]]
