"""The compiler's resource report for the 128-row attention kernels: three workgroups per CU, nothing in scratch memory."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_three_workgroups_per_cu_and_no_scratch_memory():
    hipcc = "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    csrc = os.path.join(ROOT, "magi-1_amd", "csrc")
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-I" + os.path.join(ROOT, "include"), "-I" + csrc,
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument", "--cuda-device-only",
                        "-Rpass-analysis=kernel-resource-usage", "-c", "-o", os.devnull, os.path.join(csrc, "attn_fwd_bf16_r32.hip")],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    of = lambda what: [int(x) for x in re.findall(what + r": (\d+)", r.stderr)]
    names, scratch, vgprs, lds = re.findall(r"Function Name: (\S+)", r.stderr), of(r"ScratchSize \[bytes/lane\]"), of(" VGPRs"), of(r"LDS Size \[bytes/block\]")
    assert sum("r32_kernel" in n for n in names) == 8 and len(names) == len(scratch) == len(vgprs) == len(lds) == 9  # (and the merge)
    assert not any(scratch), dict(zip(names, scratch))
    assert max(vgprs) <= 168 and 3 * max(lds) <= 160 * 1024
