"""A program that calls hipDeviceReset between two calls of the library: the second call finds
nothing of the first and returns the same results. In a process of its own (the reset ends
everything the process has on the device)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import ctypes
import numpy as np
import cva_hjm_cuda_amd as hjm

m, swap = hjm.benchmark_market(), hjm.InterestRateSwap(1e6, 0.025, 5.0)
pf = hjm.synthetic_portfolio(24, 5, seed=4)


def results():
    out = []
    for precision in (hjm.FP64, hjm.FP32_KAHAN):
        r = hjm.simulate_reference(m, swap, 3000, seed=3, precision=precision)
        out += [r.sums]
        g = hjm.cva_greeks(m, swap, 1000, seed=3, precision=precision)
        out += [g.d_spot, g.d_vol]
        p = hjm.simulate_portfolio(m, pf, 2000, seed=5, precision=precision)
        out += [p.expected_exposure, p.pfe]
    c = hjm.calibrate_pca(hjm.synthetic_history(m.volatilities, 80, seed=1), window=60, step=5, nwindows=5)
    return out + [c.eigenvalues, c.volatilities]


first = results()
path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
hip = ctypes.CDLL(path)
for i in range(2):
    assert hip.hipDeviceReset() == 0
    print("[gpu] reset", i, flush=True)
    assert all(np.array_equal(a, b) for a, b in zip(first, results()))
print("same", flush=True)
"""


@pytest.mark.gpu
def test_calls_after_a_device_reset():
    r = subprocess.run([sys.executable, "-u", "-c", PROGRAM], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("same"), r.stdout + r.stderr
