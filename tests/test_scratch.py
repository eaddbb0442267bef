"""Sizes of device scratch where an allocation fails or a limit is met: host
code of the library, linked into a small program that launches nothing."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "rtt-spgemm_amd")
HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_scratch(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "scratch")
    lib = os.path.join(PKG, "lib")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc", "hip"),
                    os.path.join(ROOT, "tests", "native", "scratch.hip"), "-o", exe,
                    "-L" + lib, "-lrtt_spgemm", "-Wl,-rpath," + lib], check=True)
    got = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                         timeout=60)
    assert got.returncode == 0, got.stdout
