"""The pinned-chunk copies (mdp_amd/csrc/host_copy.cpp) on the CPU, against played HIP calls (host_copies_cpu.cpp): every
size around the limits they are cut at, byte for byte; what has to hold when a call fails and when several engines, on one device
or two, copy at once.
"""
import os
import subprocess

import pytest

from conftest import ROOT

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_copies") / "host_copies_cpu")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host_copies_cpu.cpp"),
                    os.path.join(ROOT, "mdp_amd", "csrc", "host_copy.cpp"), "-o", out], check=True, timeout=120)
    return out


@pytest.mark.parametrize("what", ["bytes", "unwind", "two_engines", "two_devices"])
def test_host_copies(program, what):
    r = subprocess.run([program, what], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
