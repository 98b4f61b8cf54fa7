"""What the compiler makes of kernels that hold whole rows or tiles in
registers: none may keep part of them in scratch memory instead, and none whose
waits count memory instructions may have flat ones, which LDS waits wait for too
and which need not end in order."""

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


@pytest.mark.parametrize("source", [
    "tile_gemm.hip", "moe_wide.hip", "prefill_attention.hip", "seqmix_sink.hip"])
def test_no_flat_accesses_beside_counted_waits(source, tmp_path):
    hipcc, command = compile_command("_C")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    asm = tmp_path / "kernels.s"
    subprocess.run(
        command + ["--cuda-device-only", "-S", os.path.join(CSRC, source),
                   "-o", str(asm)], capture_output=True, check=True)
    text = asm.read_text()
    assert re.search(r"s_waitcnt vmcnt\([1-9]", text)
    assert not re.findall(r"\bflat_(?:load|store|atomic)\w*", text)
