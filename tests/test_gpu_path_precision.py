"""Precision of the matrix-core FP32 paths against the FP64 run on the same normals.

Tolerances, relative to the rms of a slot's forwards (ln y: of its integrals):
  * one block (1y): the forward is rounded once, when the block's sums are added up; the initial
    curve's rounding and the truncation of the small sums stay below that. 2^-24, the unit
    roundoff, bounds the rms (a rounding's own rms is less than half of it). Sums in which the
    shocks' leading products share the curve's accumulator exceed it;
  * b blocks: independent roundings of either sign add up to sqrt(b) of that, and the
    rounding of the initial curve and of the map is common to all blocks: twice sqrt(b) 2^-24.
"""
import math

import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


def _rms(expiry, paths, seed, spot=1.0, vol=1.0):
    m = hjm.benchmark_market()
    vols = vol * m.volatilities
    m = hjm.Market(spot * m.spot_rates, hjm.hjm_drift(vols), vols, m.accrual)
    swap = hjm.InterestRateSwap(1e6, 0.025, expiry)
    kw = dict(seed=seed, keep_paths=True)
    a = hjm.simulate_reference(m, swap, paths, precision=hjm.FP64, **kw)
    b = hjm.simulate_reference(m, swap, paths, precision=hjm.FP32_KAHAN,
                               path_kernel=hjm.KERNEL_MATRIX, **kw)
    slots = slice(2, int(round(2 * expiry)) + 1)

    def rel(x, y):
        return np.sqrt(((x - y) ** 2).mean(axis=0) / (y ** 2).mean(axis=0))

    return (rel(b.num_x[:, slots], a.num_x[:, slots]),
            rel(np.log(b.num_y[:, slots]), np.log(a.num_y[:, slots])))


# path counts of either launch: a workgroup per N-tile, one and two N-tiles per wave
@pytest.mark.parametrize("paths", [5000, 40000, 70000])
@pytest.mark.parametrize("spot,vol", [(1.0, 1.0), (1.15, 0.9), (0.85, 1.1)])
def test_one_block_is_rounded_once(paths, spot, vol):
    print("[gpu] one block: %d paths, curve x %g, loadings x %g" % (paths, spot, vol), flush=True)
    x, lny = _rms(1.0, paths, 11, spot, vol)
    assert x.shape == (1,) and x[0] <= 2.0 ** -24
    assert lny[0] <= 2.0 ** -24


@pytest.mark.parametrize("expiry", [5.0, 10.0, 14.0])
def test_blocks_add_their_roundings(expiry):
    print("[gpu] %gy of blocks" % expiry, flush=True)
    x, lny = _rms(expiry, 20000, 13)
    blocks = np.arange(1, x.size + 1)
    # the last tenors' backward difference amplifies what reaches it; slots from 25 on
    inner = blocks < 24
    tol = 2.0 * np.sqrt(blocks) * 2.0 ** -24
    assert np.all(x[inner] <= tol[inner])
    assert np.all(lny[inner] <= tol[inner])
    assert math.sqrt(float((x[inner] ** 2).mean())) <= 1.7e-7   # without the third accumulator 1.7 .. 2.3e-7


@pytest.mark.parametrize("expiry", [15.0, 20.0, 25.0])
def test_long_runs_add_their_roundings(expiry):
    # the kernels of 6 and 7 tiles, for all slots that the backward difference does not reach
    print("[gpu] %gy of blocks" % expiry, flush=True)
    x, lny = _rms(expiry, 20000, 17)
    blocks = np.arange(1, x.size + 1)
    inner = blocks < 24
    tol = 2.0 * np.sqrt(blocks) * 2.0 ** -24
    assert np.all(x[inner] <= tol[inner])
    assert np.all(lny[inner] <= tol[inner])


@pytest.mark.parametrize("expiry", [20.0, 25.0])
@pytest.mark.parametrize("spot,vol", [(1.0, 1.0), (1.1, 0.95), (0.9, 1.05)])
def test_a_float_step_keeps_the_last_forwards(expiry, spot, vol):
    # dt = 0.01f: c = 2 dt is not 0.02, and the last tenors' map has entries of 2e-8 that carry
    # the rest of a row's sum. EE is a mean of sums of forwards less the rate, three times as
    # sensitive as a forward, whose tolerance is the one of b blocks
    print("[gpu] float step %gy, curve x %g, loadings x %g" % (expiry, spot, vol), flush=True)
    m = hjm.benchmark_market()
    vols = vol * m.volatilities
    m = hjm.Market(spot * m.spot_rates, hjm.hjm_drift(vols), vols, m.accrual)
    swap = hjm.InterestRateSwap(1e6, 0.025, expiry)
    kw = dict(seed=19, pfe_quantile=0.975, dt=float(np.float32(0.01)))
    a = hjm.simulate_reference(m, swap, 9000, precision=hjm.FP64, **kw).expected_exposure
    b = hjm.simulate_reference(m, swap, 9000, precision=hjm.FP32_KAHAN, **kw).expected_exposure
    tol = 3.0 * 2.0 * math.sqrt(2.0 * expiry) * 2.0 ** -24
    assert np.linalg.norm(b - a) <= tol * np.linalg.norm(a)
