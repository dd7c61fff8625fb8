"""FP64 path kernel with several lanes per path against the one-path-per-lane kernel.

Host-normals runs evolve one path per lane; given the generator's own normals they see the
same shocks, and both kernels take the same FP64 operations in the same order, so the
numeraires agree bit for bit. Path counts on both sides of every change of the lane count (32,
16, 8, 4 lanes) and partly filled waves; steps per date that fill, overflow and leave
remainders in the 32-step chunks of staged shocks.
"""
import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("paths,dt,expiry", [
    (1, 0.01, 25.0), (3, 0.005, 3.0), (67, 0.02, 5.0), (130, 0.5, 12.5), (65, 0.0625, 4.0),
    (2047, 0.01, 1.5), (2049, 0.01, 1.5), (4095, 0.005, 1.0), (4097, 0.02, 1.5),
    (24575, 0.1, 2.0), (24577, 0.02, 1.0), (24577, 0.1, 2.5)])
def test_lanes_equal_one_path_per_lane(paths, dt, expiry):
    print("[gpu] FP64 lanes: %d paths, dt %g, %gy" % (paths, dt, expiry), flush=True)
    m = hjm.benchmark_market()
    swap = hjm.InterestRateSwap(1e6, 0.025, expiry)
    z = hjm.generate_normals(9, paths, int(round(expiry / dt)), stride=int(round(0.5 / dt)))
    kw = dict(dt=dt, precision=hjm.FP64, keep_paths=True)
    a = hjm.simulate_reference(m, swap, paths, seed=9, **kw)
    b = hjm.simulate_reference(m, swap, paths, normals=z, **kw)
    assert np.array_equal(a.num_x, b.num_x)
    assert np.array_equal(a.num_y, b.num_y)
    assert np.array_equal(a.sums, b.sums)
