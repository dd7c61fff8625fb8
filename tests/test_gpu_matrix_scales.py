"""The matrix-core FP32 path kernel over the scales its block map adapts to.

The shock columns of the block map pass through the matrix cores as two fp16 parts times a
power of two taken from the largest shock entry and the curve, so markets from no volatility
at all to many times the benchmark's, and curves from tiny to large against their shocks,
each take another scale. Per path against the FP64 oracle on the generator's own normals.
Tolerance: a block's output is a sum of at most 27 roundings of one FP32 ulp of the largest
partial, and a 10y run chains 19 blocks; with either sign they add up to sqrt(27 * 19) ulp,
4 standard deviations of which are 88 * 2^-23 = 1.05e-5 of the run's largest forward (the
discount integral: the same of its largest forward times 10y). Losing the low fp16 part of
either operand exceeds it.
"""
import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vol,curve,paths", [(0.0, 1.0, 17), (1e-6, 1.0, 33), (1.0, 1.0, 257),
                                             (20.0, 1.0, 33), (1.0, 1e-3, 31), (1.0, 40.0, 33)])
def test_paths_at_every_scale(oracle, vol, curve, paths):
    m = hjm.benchmark_market()
    vols = vol * m.volatilities
    m = hjm.Market(curve * m.spot_rates, hjm.hjm_drift(vols), vols, m.accrual)
    print("[gpu] matrix kernel, loadings x %g, curve x %g, %d paths" % (vol, curve, paths), flush=True)
    z = hjm.generate_normals(11, paths, 1000)
    nx, ny = oracle.reference_paths(m.spot_rates, m.drifts, m.volatilities, 10.0, 0.5, 0.01, z)
    r = hjm.simulate_reference(m, hjm.InterestRateSwap(1e6, 0.025, 10.0), paths, seed=11,
                               precision=hjm.FP32_KAHAN, keep_paths=True,
                               path_kernel=hjm.KERNEL_MATRIX)
    tol = 1.05e-5 * np.max(np.abs(nx))
    assert np.max(np.abs(r.num_x - nx)) <= tol
    live = ny != 0
    assert np.max(np.abs(np.log(r.num_y[live] / ny[live]))) <= 10.0 * tol
