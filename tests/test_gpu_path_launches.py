"""Matrix-core FP32 paths at the path counts where their launches change.

Few paths take a workgroup per 16 paths, more a wave per 16, then a wave per 32; beyond a
whole turn of the chip the rest is launched by itself. Every path goes through the same
operations in the same order whichever launch takes it, so runs of any count agree bit for bit
on the paths they share (a path's shocks follow its number), and with the stored shocks' sweep.
"""
import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu

COUNTS = [1, 17, 12289, 16385, 20481, 49153, 65535, 65537, 65536 + 12289]


@pytest.mark.parametrize("paths", COUNTS)
@pytest.mark.parametrize("expiry", [1.0, 16.0, 25.0])
def test_reference_paths_do_not_depend_on_the_launch(paths, expiry):
    print("[gpu] path launches: %d paths, %gy" % (paths, expiry), flush=True)
    m = hjm.benchmark_market()
    swap = hjm.InterestRateSwap(1e6, 0.025, expiry)

    def run(count, offset):
        r = hjm.simulate_reference(m, swap, count, seed=3, precision=hjm.FP32_KAHAN, keep_paths=True,
                                   path_kernel=hjm.KERNEL_MATRIX, path_offset=offset)
        return r.num_x, r.num_y

    x, y = run(paths, 0)
    for first in {0, paths // 2, max(0, paths - 40)}:
        n = min(40, paths - first)
        a, b = run(n, first)
        assert np.array_equal(x[first:first + n], a) and np.array_equal(y[first:first + n], b)


@pytest.mark.parametrize("paths", COUNTS)
def test_portfolio_paths_do_not_depend_on_the_launch(paths):
    print("[gpu] path launches, portfolio: %d paths" % paths, flush=True)
    m = hjm.benchmark_market()
    pf = hjm.synthetic_portfolio(8, 2, seed=3)
    pf.periods = np.minimum(pf.periods, 6).astype(np.int32)

    def run(**tuning):
        return hjm.simulate_portfolio(m, pf, paths, keep_paths=True, horizon=3.0, seed=3,
                                      path_kernel=hjm.KERNEL_MATRIX, tuning=hjm.Tuning(**tuning)).exposures

    assert np.array_equal(run(), run(path_tiles=1, path_waves=16))


@pytest.mark.parametrize("paths", [12288, 16385, 49153])
def test_stored_shocks_do_not_depend_on_the_launch(paths):
    print("[gpu] path launches, stored shocks: %d paths" % paths, flush=True)
    m = hjm.benchmark_market()
    for expiry in (2.0, 17.0):
        swap = hjm.InterestRateSwap(1e6, 0.02, expiry)
        a, b = (hjm.cva_greeks(m, swap, paths, seed=5, precision=hjm.FP32_KAHAN, regenerate_normals=again)
                for again in (False, True))
        assert a.stored_normals_bytes > 0 == b.stored_normals_bytes
        for x, y in ((a.d_spot, b.d_spot), (a.d_vol, b.d_vol), (a.d_drift, b.d_drift)):
            assert np.array_equal(x, y)
