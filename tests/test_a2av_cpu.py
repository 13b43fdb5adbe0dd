"""All-to-all-v from the callers' tables, on the host: the tables that launches read in device memory, on a model of streams and events
(tests/c_abi/a2av_check.cc against csrc/a2av.cc)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("needs a host C++ compiler and the HIP headers")
    csrc = os.path.join(ROOT, "cann-hccl_amd", "csrc")
    exe = str(tmp_path_factory.mktemp("a2av") / "a2av_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-Werror", "-D__HIP_PLATFORM_AMD__", "-isystem", os.path.join(ROCM, "include"), "-I", csrc,
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "c_abi", "a2av_check.cc"), os.path.join(csrc, "a2av.cc"), "-o", exe],
                   check=True)
    return exe


# (the sets kept are eight, the streams a set remembers as many)
@pytest.mark.parametrize("ranks,calls,streams,sets", [(20, 3000, 1, 5), (20, 3000, 1, 12), (20, 3000, 3, 5), (20, 4000, 3, 12), (33, 2000, 2, 9), (40, 1500, 20, 6),
                                                      (64, 600, 2, 3), (17, 3000, 12, 10), (17, 6000, 30, 9), (12, 3000, 3, 5), (3, 3000, 3, 12)])
def test_tables_of_several_streams(check, ranks, calls, streams, sets):
    out = subprocess.run([check, str(ranks), str(calls), str(streams), str(sets)], stdout=subprocess.PIPE, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.stdout


@pytest.mark.parametrize("ranks", [2, 8, 13, 40, 64])
def test_calls_that_go_the_general_way(check, ranks):
    out = subprocess.run([check, str(ranks), "0"], stdout=subprocess.PIPE, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.stdout


@pytest.mark.parametrize("ranks", [2, 16, 17, 64])
def test_widths(check, ranks):
    out = subprocess.run([check, str(ranks), "-1"], stdout=subprocess.PIPE, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.stdout
