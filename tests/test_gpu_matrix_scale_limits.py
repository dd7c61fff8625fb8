"""The matrix-core FP32 paths at the limits of the block map's scale, against the FP64 oracle.

Loadings next to nothing beside a large curve over 25 years: the scale follows the curve there, and
the integrals stay finite. Tolerance as for the other scales: 27 roundings a block and 49
blocks of either sign, 4 sqrt(27 x 49) 2^-23 of the largest forward, 25 times that of ln y.

Loadings that differ by 24 binades between the tenors on a curve of zeros, tenor by tenor: a
slot's forward has 88 roundings of 2^-23 of its own largest value (4 sqrt(27 x 19), 10 years), and
the map's entries an absolute error of 2^-37 of the largest one, over 150 shocks of each of
19 blocks: 4 sqrt(150 x 19) 2^-37.
"""
import math

import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


def _run(oracle, m, expiry, paths):
    z = hjm.generate_normals(11, paths, int(round(expiry / 0.01)))
    nx, ny = oracle.reference_paths(m.spot_rates, m.drifts, m.volatilities, expiry, 0.5, 0.01, z)
    r = hjm.simulate_reference(m, hjm.InterestRateSwap(1e6, 0.025, expiry), paths, seed=11,
                               precision=hjm.FP32_KAHAN, keep_paths=True, path_kernel=hjm.KERNEL_MATRIX)
    return nx, ny, r.num_x, r.num_y


@pytest.mark.parametrize("vol", [1e-30, 1e-40, 1e-44])
def test_loadings_next_to_nothing(oracle, vol):
    m = hjm.benchmark_market()
    vols = vol * m.volatilities
    m = hjm.Market(20.0 * m.spot_rates, hjm.hjm_drift(vols), vols, m.accrual)
    print("[gpu] loadings x %g beside a curve x 20, 25y" % vol, flush=True)
    nx, ny, x, y = _run(oracle, m, 25.0, 17)
    tol = 4.0 * math.sqrt(27 * 49) * 2.0 ** -23 * np.max(np.abs(nx))
    assert np.max(np.abs(x - nx)) <= tol
    live = ny != 0
    assert np.all(np.isfinite(y)) and np.all(y[live] > 0)
    assert np.max(np.abs(np.log(y[live] / ny[live]))) <= 25.0 * tol


@pytest.mark.parametrize("rising", [False, True])
def test_loadings_many_binades_apart(oracle, rising):
    m = hjm.benchmark_market()
    span = np.linspace(-24.0, 0.0, hjm.TENORS) if rising else np.linspace(0.0, -24.0, hjm.TENORS)
    vols = np.array([[0.01], [-0.006], [0.004]]) * 2.0 ** span
    m = hjm.Market(np.zeros(hjm.TENORS), hjm.hjm_drift(vols), vols, m.accrual)
    print("[gpu] loadings over 24 binades, %s, on zeros" % ("rising" if rising else "falling"), flush=True)
    nx, _, x, _ = _run(oracle, m, 10.0, 65)
    top = np.max(np.abs(hjm.block_map(m)[:, 64:]))
    slots = slice(2, 21)
    tol = 88.0 * 2.0 ** -23 * np.max(np.abs(nx[:, slots]), axis=0) + 4.0 * math.sqrt(150 * 19) * 2.0 ** -37 * top
    assert np.all(np.max(np.abs(x[:, slots] - nx[:, slots]), axis=0) <= tol)
