"""What the library does on the host - memory kept, copies, closing and opening it on another device - with a stand-in for
the HIP runtime (host_runtime.cpp): no GPU is needed, and there are two."""
import os
import subprocess

import pytest

from comet_amd import runtime as rt

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    rt.lib()          # built
    exe = str(tmp_path_factory.mktemp("host_runtime") / "main")
    lib = os.path.join(ROOT, "comet_amd")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-isystem", f"{ROCM}/include", "-I",
                           os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host_runtime.cpp"), "-o", exe,
                           os.path.join(lib, "libcomet_hip_rt.so"), f"-Wl,-rpath,{lib}", f"-Wl,-rpath-link,{ROCM}/lib",
                           "-Wl,--allow-shlib-undefined", "-lpthread", "-ldl"])
    return exe


@pytest.mark.parametrize("scenario", ["another_device", "whole_device", "given_back", "block_of_another_device",
                                      "memory_while_another_waits", "waiting_is_cheap", "no_threads", "two_threads", "refused_launch"])
def test_host_side(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
