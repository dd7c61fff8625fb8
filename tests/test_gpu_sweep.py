"""The matrix-core reverse sweep against the oracle's FP64 adjoint.

Sizes where it changes shape: paths that leave its waves, 32-path units and workgroups partly
filled; horizons on both sides of every number of row tiles (mu rows to dates 15, 31, 47, 50)
and the one-block horizon. Seeds and sweep are FP32 with the paths' terms of
either sign: 2e-5 of a gradient's scale covers sqrt(25 y x 50 steps) roundings of 2^-24 with a
factor of ten. Shocks stored by the forward or regenerated in bounded chunks give the same
sums bit for bit. FP64 runs keep the one-pass VALU sweep, with or without stored shocks.
"""
import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


def _close(got, want):
    for g, w in zip(got, want):
        assert np.max(np.abs(g - w)) <= 2e-5 * np.max(np.abs(w))


@pytest.mark.parametrize("paths,expiry", [(1, 1.0), (3, 7.5), (31, 8.0), (33, 15.5), (129, 16.0),
                                          (65, 23.5), (40, 24.0), (257, 25.0)])
def test_reference_sweep_matches_oracle(oracle, paths, expiry):
    print("[gpu] matrix sweep: %d paths, %gy" % (paths, expiry), flush=True)
    m = hjm.benchmark_market()
    z = hjm.generate_normals(5, paths, int(round(expiry / 0.01)))
    w = hjm.cva_weights(0.02, 0.4)
    cva, ds, dv, dm = oracle.reference_cva_greeks(m.spot_rates, m.drifts, m.volatilities, m.accrual,
                                                  1e6, 0.02, expiry, 0.5, 0.01, z, w)
    swap = hjm.InterestRateSwap(1e6, 0.02, expiry)
    a = hjm.cva_greeks(m, swap, paths, seed=5, precision=hjm.FP64)
    d = hjm.cva_greeks(m, swap, paths, seed=5, precision=hjm.FP64, path_kernel=hjm.KERNEL_MATRIX)
    b = hjm.cva_greeks(m, swap, paths, seed=5, precision=hjm.FP32_KAHAN)
    c = hjm.cva_greeks(m, swap, paths, seed=5, precision=hjm.FP32_KAHAN, regenerate_normals=True)
    assert a.stored_normals_bytes == c.stored_normals_bytes == 0
    assert b.stored_normals_bytes > 0 and d.stored_normals_bytes > 0
    for g in (a, d):
        assert g.cva == pytest.approx(cva, rel=1e-9)
    for g in (a, b, d):
        _close((g.d_spot, g.d_vol, g.d_drift), (ds, dv, dm))
    for x, y in ((b.d_spot, c.d_spot), (b.d_vol, c.d_vol), (b.d_drift, c.d_drift)):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("paths,horizon", [(1, 0.5), (33, 2.0), (127, 30.0)])
def test_portfolio_sweep_matches_oracle(oracle, paths, horizon):
    print("[gpu] matrix sweep, portfolio: %d paths, %gy" % (paths, horizon), flush=True)
    m = hjm.benchmark_market()
    pf = hjm.synthetic_portfolio(20, 4, seed=3)
    pf.periods = np.minimum(pf.periods, int(2 * horizon)).astype(np.int32)
    z = hjm.generate_normals(5, paths, int(round(horizon / 0.01)))
    w = oracle.portfolio_weights(pf, horizon)
    cva, ds, dv, dm = oracle.portfolio_cva_greeks(m.spot_rates, m.drifts, m.volatilities, horizon, 0.5,
                                                  0.01, z, pf, w)
    a = hjm.portfolio_cva_greeks(m, pf, paths, horizon=horizon, seed=5, precision=hjm.FP64)
    d = hjm.portfolio_cva_greeks(m, pf, paths, horizon=horizon, seed=5, precision=hjm.FP64,
                                 path_kernel=hjm.KERNEL_MATRIX)
    b = hjm.portfolio_cva_greeks(m, pf, paths, horizon=horizon, seed=5, precision=hjm.FP32_KAHAN)
    for g in (a, d):
        assert g.cva == pytest.approx(cva, rel=1e-8)
    for g in (a, b, d):
        _close((g.d_spot, g.d_vol, g.d_drift), (ds, dv, dm))
