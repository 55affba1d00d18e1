"""The library's host code on a device of host memory (tests/cxx/host_device.cpp):
error paths and the use of device memory, without a GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_device") / "host_device")
    lib = os.path.join(ROOT, "mrchem_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-rdynamic",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(lib, "csrc"),
                    "-isystem", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
                    os.path.join(ROOT, "tests", "cxx", "host_device.cpp"), "-o", out, "-L" + lib, "-lmwgreen",
                    "-Wl,-rpath," + lib], check=True)
    return out


@pytest.mark.parametrize("scenario", ["split_step_fails", "idle_memory_is_given_back", "idle_memory_is_bounded",
                                      "host_output_memory", "apply_stages", "more_than_a_launch"])
def test_scenario(exe, scenario):
    r = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr)
    assert r.returncode == 0, r.stdout + r.stderr
