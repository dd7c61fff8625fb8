"""The reverse sweep's portions, segments and buffers, on the CPU: the host code that launches it,
compiled with the host compiler over a stand-in for the HIP runtime (tests/cpp/fake_hip)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cva_hjm_cuda_amd", "csrc")
CPP = os.path.join(ROOT, "tests", "cpp")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("sweep") / "sweep_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-pthread",
                    "-I" + os.path.join(CPP, "fake_hip"), "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                    "-o", exe, os.path.join(CPP, "sweep_driver.cpp"),
                    "-x", "c++", os.path.join(CSRC, "hjm_pool.hip")], check=True)
    return exe


@pytest.mark.parametrize("check", ["portions_cover_every_path_once", "memory_that_does_not_suffice"])
def test_sweep(driver, check):
    r = subprocess.run([driver, check], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
