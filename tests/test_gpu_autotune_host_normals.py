"""The autotuner on FP64 plans with host normals, whose path kernel has launch shapes: accepted for
any horizon (one date interval included, where the two-date tuning run must not read past the
caller's normals) and any path kernel, and its choice changes no result."""
import ctypes as C

import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm
from cva_hjm_cuda_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("horizon,kernel", [(0.5, hjm.KERNEL_AUTO), (3.0, hjm.KERNEL_AUTO),
                                            (3.0, hjm.KERNEL_VECTOR), (3.0, hjm.KERNEL_MATRIX)])
def test_fp64_host_normals(horizon, kernel):
    paths = 700
    print("[gpu] autotune, FP64 host normals, %gy, path kernel %d" % (horizon, kernel), flush=True)
    m = hjm.benchmark_market()
    pf = hjm.synthetic_portfolio(8, 2, seed=3)
    pf.periods = np.minimum(pf.periods, int(2 * horizon)).astype(np.int32)
    z = hjm.generate_normals(9, paths, int(round(horizon / 0.01)))
    mk, pfc = m._c(), api._pf_c(pf, horizon, 0.4)
    cfg = api._config(paths, 0.01, hjm.FP64, api.RNG_HOST, 9, z, 0.0, 0.4, 0.975, 0, 0, kernel)
    t, ms = api._Tuning(), C.c_double()
    assert api.library().hjm_portfolio_autotune(C.byref(mk), C.byref(pfc), C.byref(cfg), C.byref(t),
                                                C.byref(ms)) == 0
    tuning = hjm.Tuning._from_c(t)
    assert ms.value > 0 and tuning.block_size in (64, 128, 256) and tuning.use_graph
    kw = dict(horizon=horizon, precision=hjm.FP64, seed=9, normals=z)
    a, b = (hjm.simulate_portfolio(m, pf, paths, tuning=u, **kw) for u in (None, tuning))
    assert np.array_equal(a.expected_exposure, b.expected_exposure) and np.array_equal(a.pfe, b.pfe)
