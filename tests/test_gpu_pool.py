"""Device memory kept between calls: results do not depend on what earlier calls left in it,
with one thread or several, before and after it is given back."""
import threading

import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu


def _calls():
    m = hjm.benchmark_market()
    pf = hjm.synthetic_portfolio(24, 5, seed=4)

    def reference(paths, expiry, precision):
        r = hjm.simulate_reference(m, hjm.InterestRateSwap(1e6, 0.025, expiry), paths, seed=3,
                                   precision=precision, keep_paths=True, pfe_quantile=0.0)
        return [r.sums, r.num_x, r.num_y, r.exposures]

    def greeks(precision):
        g = hjm.cva_greeks(m, hjm.InterestRateSwap(1e6, 0.025, 3.0), 513, seed=3, precision=precision)
        return [np.array([g.cva, g.cva_stderr]), g.d_spot, g.d_vol, g.d_drift, g.d_vol_total]

    def portfolio(precision):
        r = hjm.simulate_portfolio(m, pf, 600, keep_paths=True, seed=5, precision=precision)
        return [r.expected_exposure, r.pfe, r.cva, r.cva_stderr, r.exposures]

    def portfolio_greeks(precision):
        g = hjm.portfolio_cva_greeks(m, pf, 600, seed=5, precision=precision)
        return [np.array([g.cva]), g.d_spot, g.d_vol, g.d_drift, g.d_vol_total]

    out = []
    for prec in (hjm.FP64, hjm.FP32_KAHAN):
        out += [lambda p=prec: reference(700, 10.0, p), lambda p=prec: reference(699, 2.0, p),
                lambda p=prec: greeks(p), lambda p=prec: portfolio(p),
                lambda p=prec: portfolio_greeks(p)]
    return out


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def test_reused_memory_and_threads_do_not_change_results():
    calls = _calls()
    fresh = []
    for i, c in enumerate(calls):
        print("[gpu] pool: call %d on fresh memory" % i, flush=True)
        hjm.release_cached_memory()
        fresh.append(c())
    for i in list(range(len(calls))) + list(reversed(range(len(calls)))):
        assert _same(calls[i](), fresh[i]), i
    print("[gpu] pool: four threads", flush=True)
    bad = []

    def work(start):
        for k in range(len(calls)):
            i = (start + 3 * k) % len(calls)
            try:
                if not _same(calls[i](), fresh[i]):
                    bad.append(i)
            except Exception as e:   # noqa: BLE001 (a thread's failure fails the test)
                bad.append(e)
            if k == 4:
                hjm.release_cached_memory()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
