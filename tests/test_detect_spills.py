"""The FP32 detect of many users at 32 antennas keeps its accumulators in registers (compiled for gfx950, no GPU): with
more than a few spilled it is slower than the FP32 matrix instructions it replaced."""
import os
import re
import subprocess

from conftest import ROOT


def test_many_users_do_not_spill(tmp_path):
    out = str(tmp_path / "spills.s")
    subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only", "-S", "-w",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I" + os.path.join(ROOT, "libapsm_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "detect_spills.hip"), "-o", out],
                   check=True)
    spilled = [int(n) for n in re.findall(r"\.vgpr_spill_count:\s*(\d+)", open(out).read())]
    assert len(spilled) == 2 and max(spilled) < 32, spilled
