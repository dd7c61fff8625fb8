"""Portfolios of few paths: FP64 paths with several lanes per path, statistics of one path per
thread.

FP64 paths against the one-path-per-lane kernel, which host-supplied normals still take: the
same operations in the same order, so results agree bit for bit at every lane count and ragged
path count. The statistics against the exposures of the same run in numpy: FP64 sums of up to
P values per date and, for CVA, dates, 2e-12 relative.
"""
import math

import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("paths,horizon,dt", [(1, 3.0, 0.01), (2048, 1.0, 0.01), (2049, 1.0, 0.01),
                                              (4097, 1.0, 0.05), (24577, 1.0, 0.025), (70, 30.0, 0.01)])
def test_fp64_paths_take_the_same_values(paths, horizon, dt):
    print("[gpu] FP64 portfolio paths: %d paths, %gy, dt %g" % (paths, horizon, dt), flush=True)
    m = hjm.benchmark_market()
    pf = hjm.synthetic_portfolio(8, 2, seed=3)
    pf.periods = np.minimum(pf.periods, int(2 * horizon)).astype(np.int32)
    stride = int(round(0.5 / dt))
    z = hjm.generate_normals(9, paths, int(round(horizon / dt)), stride=stride)
    kw = dict(horizon=horizon, dt=dt, precision=hjm.FP64, seed=9)
    a = hjm.simulate_portfolio(m, pf, paths, keep_paths=True, **kw)
    b = hjm.simulate_portfolio(m, pf, paths, keep_paths=True, normals=z, **kw)
    assert np.array_equal(a.exposures, b.exposures)


@pytest.mark.parametrize("precision", ["FP32_KAHAN", "FP64"])
@pytest.mark.parametrize("paths,sets,horizon", [(1, 1, 0.5), (255, 3, 3.5), (257, 2, 30.0), (393216, 1, 1.0),
                                                (393217, 1, 1.0), (4097, 2, 4.0)])
def test_statistics_of_the_exposures(paths, sets, horizon, precision):
    print("[gpu] portfolio statistics: %d paths x %d sets, %gy, %s" % (paths, sets, horizon, precision),
          flush=True)
    m = hjm.benchmark_market()
    pf = hjm.synthetic_portfolio(max(3, sets), sets, seed=3)
    pf.periods = np.minimum(pf.periods, int(2 * horizon)).astype(np.int32)
    r = hjm.simulate_portfolio(m, pf, paths, keep_paths=True, horizon=horizon, seed=9, pfe_quantile=0.0,
                               precision=getattr(hjm, precision))
    e = np.asarray(r.exposures, np.float64)
    # exactly rounded sums (numpy's own over the leading axis adds row by row, 6e-12 off here)
    want = np.array([[math.fsum(e[:, g, d]) / paths for d in range(e.shape[2])] for g in range(sets)])
    assert np.max(np.abs(np.asarray(r.expected_exposure).reshape(want.shape) - want)) <= 2e-12 * max(
        np.max(want), 1e-300)
