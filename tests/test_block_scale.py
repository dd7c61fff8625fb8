"""The power of two in the FP32 block map, on the CPU: the largest shock entry at most 2^13 (fp16's
range), the curve under 2^40 for any loadings, next to none included, and both where they are
meant to be for ordinary markets."""
import os
import subprocess

import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("scale") / "block_scale_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra",
                    "-I" + os.path.join(ROOT, "tests", "cpp", "fake_hip"), "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "cva_hjm_cuda_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "block_scale_driver.cpp")], check=True)
    return exe


def test_scale_keeps_curve_and_shocks_in_range(driver):
    m = hjm.benchmark_market()
    cases = [(c, v, d, pf) for c in (0.0, 1e-30, 1e-3, 1.0, 40.0, 1e6)
             for v in (0.0, 1e-45, 1e-30, 1e-12, 1e-6, 1.0, 1e3, 1e9) for d in (0.0, 1e-4) for pf in (0, 1)]
    text = " ".join("%.17g" % x for x in np.concatenate([m.spot_rates, np.ravel(m.volatilities)])) + "\n"
    text += "\n".join("%.17g %.17g %.17g %d" % c for c in cases)
    out = subprocess.run([driver], input=text, capture_output=True, text=True, check=True).stdout
    got = np.array([line.split() for line in out.splitlines()], float)
    assert got.shape == (len(cases), 3)
    for (c, v, d, _), (k, top, high) in zip(cases, got):
        assert top < 2.0 ** 13 and high < 2.0 ** 40, (c, v, d, k, top, high)
        if v == 0.0 and d == 0.0:
            assert k == 0
        elif abs(k) < 120 and high < 2.0 ** 39:   # neither bound is met
            assert top >= 2.0 ** 12, (c, v, d, k, top, high)
