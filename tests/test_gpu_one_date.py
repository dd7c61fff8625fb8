"""A run of a single exposure date evolves nothing: slot 1 holds the initial curve's tenor 1 and the
frozen half year's discount factor on every path, in either precision, at ragged path counts and
those of every launch shape."""
import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["FP64", "FP32_KAHAN"])
@pytest.mark.parametrize("paths", [1, 257, 5000, 66001])
def test_single_date(paths, precision):
    print("[gpu] one date: %d paths, %s" % (paths, precision), flush=True)
    m = hjm.benchmark_market()
    r = hjm.simulate_reference(m, hjm.InterestRateSwap(1e6, 0.005, 0.5), paths, seed=9, keep_paths=True,
                               precision=getattr(hjm, precision))
    f = m.spot_rates[1]
    x = f if precision == "FP64" else np.float64(np.float32(f))
    assert np.all(r.num_x[:, 1] == x)
    # 50 additions of the curve (as the precision holds it) and one exponential
    assert np.max(np.abs(r.num_y[:, 1] / np.exp(-0.5 * x) - 1.0)) <= 1e-14
    assert np.all(r.num_x[:, 2:] == 0) and np.all(r.exposures[:, 1:] == 0)
    assert r.expected_exposure[0] > 0
