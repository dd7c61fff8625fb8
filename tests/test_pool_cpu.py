"""The cache of device memory and plan contexts, on the CPU: its host code compiled with the
host compiler over a stand-in for the HIP runtime (tests/cpp/fake_hip)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cva_hjm_cuda_amd", "csrc")
CPP = os.path.join(ROOT, "tests", "cpp")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pool") / "pool_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-pthread",
                    "-I" + os.path.join(CPP, "fake_hip"), "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                    "-o", exe, os.path.join(CPP, "pool_driver.cpp"),
                    "-x", "c++", os.path.join(CSRC, "hjm_pool.hip")], check=True)
    return exe


@pytest.mark.parametrize("check", ["blocks_of_a_failed_stream", "pinned_buffers_that_cannot_be_had",
                                   "memory_close_to_the_cards", "a_device_reset"])
def test_pool(driver, check):
    r = subprocess.run([driver, check], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
