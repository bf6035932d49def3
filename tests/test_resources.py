"""What the compiler gives the kernels whose speed depends on the workgroups a CU
holds: registers and scratch from its resource remarks (no device needed)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "npu880-mtk-npu-llm-runtime_amd")
HIPCC = "/opt/rocm/bin/hipcc"


def _resources(source):
    """{kernel: (waves per SIMD, scratch bytes)} with the Makefile's own flags."""
    r = subprocess.run(["make", "-s", "-C", PKG, "print-flags"], capture_output=True, text=True, timeout=60, check=True)
    out = subprocess.run([HIPCC, *r.stdout.split(), "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                          os.path.join(PKG, "csrc", source), "-o", os.devnull],
                         capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr[-2000:]
    got = {}
    for part in out.stderr.split("Function Name: ")[1:]:
        num = {k: int(re.search(re.escape(k) + r": (\d+)", part).group(1))
               for k in ("ScratchSize [bytes/lane]", "Occupancy [waves/SIMD]")}
        got[part.split()[0]] = (num["Occupancy [waves/SIMD]"], num["ScratchSize [bytes/lane]"])
    return got


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
def test_rmsnorm_four_workgroups_per_cu():
    """Every width of the RMSNorm producer leaves registers for four workgroups
    of 256 threads (a wave on each SIMD) per CU, without scratch."""
    rms = {k: v for k, v in _resources("qmm_quant.hip").items() if "rmsnorm_q8k_kernel" in k}
    assert len(rms) == 5
    for name, (waves, scratch) in rms.items():
        assert waves >= 4 and scratch == 0, (name, waves, scratch)
