"""The executor's rules on sizes and alignment, on the host (tests/c_abi/launch_rules_check.cc against csrc/launch_rules.h)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_rules(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("needs a host C++ compiler")
    exe = str(tmp_path / "launch_rules_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "cann-hccl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "c_abi", "launch_rules_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "OK", out.stdout
