"""Precision of FP32 books: EE and PFE against the FP64 run on the same normals.

The measure is the 2-norm of the error over all sets and dates relative to the result's, averaged
over six random books. `former` is what the valuation held when every product was accumulated,
one after another, from the set's constant on (three bf16 parts per shock in the paths); sums that
drop bits at the size of the gross book hold 1.2 to 3 times that in PFE. A tenth on top of it for
the spread of an average of six.
"""
import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sets,swaps,paths,horizon,former", [
    (3, 20, 2000, 10.0, (5.32e-7, 4.78e-7)),
    (11, 57, 10007, 30.0, (3.90e-7, 3.01e-7)),
    (32, 256, 20000, 20.0, (3.47e-7, 3.01e-7)),
    (64, 300, 5000, 30.0, (3.62e-7, 3.26e-7)),
    (128, 1024, 4000, 30.0, (3.43e-7, 3.49e-7)),
    (8, 40, 65536, 20.0, (5.82e-7, 3.64e-7)),
    (6, 30, 262144, 10.0, (4.41e-7, 4.04e-7)),
    (5, 12, 262144, 30.0, (4.39e-7, 3.23e-7)),
])
def test_books_are_as_close_to_fp64_as_before(sets, swaps, paths, horizon, former):
    m = hjm.benchmark_market()
    err = []
    for seed in range(1, 7):
        print("[gpu] book of %d swaps in %d sets, %d paths x %gy, seed %d"
              % (swaps, sets, paths, horizon, seed), flush=True)
        pf = hjm.synthetic_portfolio(swaps, sets, seed=1000 * sets + seed)
        pf.periods = np.minimum(pf.periods, int(2 * horizon)).astype(np.int32)
        kw = dict(seed=20 + seed, pfe_quantile=0.975, horizon=horizon)
        a = hjm.simulate_portfolio(m, pf, paths, precision=hjm.FP64, **kw)
        b = hjm.simulate_portfolio(m, pf, paths, precision=hjm.FP32_KAHAN, **kw)
        err.append([np.linalg.norm(x - y) / np.linalg.norm(y)
                    for x, y in ((b.expected_exposure, a.expected_exposure), (b.pfe, a.pfe))])
    ee, pfe = np.mean(err, axis=0)
    assert ee <= 1.1 * former[0]
    assert pfe <= 1.1 * former[1]
