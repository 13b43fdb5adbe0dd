"""Small collectives, whose descriptors ride in the kernel arguments, on the host: which calls go that way, and that the
arguments say what the plan says (tests/c_abi/direct_check.cc against csrc/direct.cc and the planner)."""
import os
import shutil
import subprocess

import pytest

from hccl_loader import load

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_the_arguments_are_the_plans_items(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("needs a host C++ compiler and the HIP headers")
    csrc = os.path.join(ROOT, "cann-hccl_amd", "csrc")
    exe = str(tmp_path / "direct_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-Werror", "-D__HIP_PLATFORM_AMD__", "-isystem", os.path.join(ROCM, "include"), "-I", csrc,
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "c_abi", "direct_check.cc"),
                    *[os.path.join(csrc, f) for f in ("direct.cc", "plan.cc", "plan_schedules.cc", "plan_lower.cc", "plan_fuse.cc", "plan_template.cc")],
                    "-o", exe], check=True)
    out = subprocess.run([exe, "20000"], stdout=subprocess.PIPE, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.stdout
    # every kind of record was met, and every reason to go another way
    assert min(int(w) for w in out.stdout.split() if w.isdigit()) > 500, out.stdout


def test_the_setting():
    H = load()
    comms = H.comm_init_all(2)
    for v in ("0", "auto"):
        H.set_param(comms[0], "direct", v)
    for v in ("1", "2", "", "yes"):
        with pytest.raises(H.HcclError) as e:
            H.set_param(comms[0], "direct", v)
        assert e.value.code == H.HCCL_E_PARA
    assert H.last_op_info(comms[0])["direct"] == 0
    H.comm_destroy(comms)
