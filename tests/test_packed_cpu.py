"""The packed arguments of small collectives, on the host: read back as the kernels read them, they are the plan's items
(tests/c_abi/packed_check.cc against csrc/direct.cc and the planner)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_the_packed_arguments_are_the_plans_items(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("needs a host C++ compiler and the HIP headers")
    csrc = os.path.join(ROOT, "cann-hccl_amd", "csrc")
    exe = str(tmp_path / "packed_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-Werror", "-D__HIP_PLATFORM_AMD__", "-isystem", os.path.join(ROCM, "include"), "-I", csrc,
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "c_abi", "packed_check.cc"),
                    *[os.path.join(csrc, f) for f in ("direct.cc", "plan.cc", "plan_schedules.cc", "plan_lower.cc", "plan_fuse.cc", "plan_template.cc")],
                    "-o", exe], check=True)
    out = subprocess.run([exe, "10000"], stdout=subprocess.PIPE, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.stdout
    # every size of arguments was met, trees, buffers in place and too far apart, and items that are not alike
    assert min(int(w) for w in out.stdout.split() if w.isdigit() and w not in ("8", "16", "32")) > 200, out.stdout
