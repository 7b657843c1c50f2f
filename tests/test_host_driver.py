"""The host side of the solver over a stand-in HIP runtime (no GPU): what it
does when an allocation fails, and what it hands to the kernels."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = tmp_path_factory.mktemp("host_driver") / "driver"
    src = os.path.join(ROOT, "cup3d_amd", "csrc")
    r = subprocess.run(
        ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
         os.path.join(ROOT, "include"), "-I", src,
         os.path.join(ROOT, "tests", "host_driver", "driver.cpp"),
         os.path.join(src, "topology.cpp"), "-o", str(exe), "-pthread", "-no-pie",
         "-Wl,--unresolved-symbols=ignore-all"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("scenario", ["failed_allocations", "volume", "growing_meshes",
                                      "timed_diffusion_kernels"])
def test_scenario(driver, scenario):
    r = subprocess.run([str(driver), scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
