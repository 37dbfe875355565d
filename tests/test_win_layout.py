"""The window sequencer's block buffers hold every float its copies and loads read (host side, no GPU)."""
import os
import subprocess

from conftest import ROOT


def test_reads_stay_inside_the_reserved_buffers(tmp_path):
    exe = str(tmp_path / "win_layout_check")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-Wno-unused",
                    "-I" + os.path.join(ROOT, "libapsm_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "win_layout_check.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert "0 windows with reads out of range" in r.stdout
