"""A server's progress step uploads few frames ahead, also where every copy holds the host (no GPU)."""
import os
import subprocess

from conftest import ROOT


def test_a_step_uploads_two_frames_at_most(tmp_path):
    exe = str(tmp_path / "serve_ahead_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-I" + os.path.join(ROOT, "libapsm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "serve_ahead_check.cpp"), "-o", exe], check=True)
    pageable, pinned, single, large, full = map(int, subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split())
    assert pageable == 2 and pinned == 2  # without the limit a pageable step takes all 64 MB
    assert single == 1 and large == 1 and full == 0
