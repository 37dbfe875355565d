"""The inline copies to LDS tell the compiler that they change M0 (compiled for gfx950, no GPU)."""
import os
import re
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("m0") / "probe.s")
    subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only", "-S", "-w",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I" + os.path.join(ROOT, "libapsm_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "m0_probe.hip"), "-o", out],
                   check=True)
    return open(out).read()


@pytest.mark.parametrize("kernel", ["probe_dword", "probe_dwordx4"])
def test_m0_is_set_again_after_an_inline_copy(assembly, kernel):
    body = re.search(rf"^{kernel}:(.*?)s_endpgm", assembly, re.S | re.M).group(1)
    before, after = body.split("#ASMEND")
    assert "load_lds" in before.split("#ASMSTART")[0] and "load_lds" in after
    assert re.search(r"m0,", after.split("load_lds")[0])
