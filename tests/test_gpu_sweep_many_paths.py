"""The matrix-core reverse sweep at path counts far beyond one turn of the chip.

Its FP32 sums cover a bounded number of paths and meet in FP64, so a run's gradients are the
average of its slices' whatever its length: slices of whole workgroups give the same FP32 sums, and
8192 FP64 additions in another order move an average by less than 1e-10 of the largest component.
Against the FP64 run (whose one-pass sweep adds up to two blocks in FP32) 3e-6 of a gradient's
2-norm: sqrt(2 x 50 x 2^15) roundings of 2^-24 of a term, over as many terms, are under 1e-9 of the
sum; what is left is either sweep's own recursion over 900 steps, 900 x 2^-24 / sqrt(900) = 1.8e-6,
and as much again for the forward paths.
Stored and regenerated shocks pass in different portions and give the same sums bit for bit: over
2^30 bytes of regenerated shocks (60001 paths x 17y, with a ragged last portion) and over a segment
of 4096 workgroups (600001 paths).
"""
import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu

FIELDS = ("d_spot", "d_vol", "d_drift", "d_vol_total")


def _deal(paths, expiry, precision=hjm.FP32_KAHAN, **kw):
    print("[gpu] deal Greeks: %d paths x %gy %s" % (paths, expiry, kw), flush=True)
    return hjm.cva_greeks(hjm.benchmark_market(), hjm.InterestRateSwap(1e6, 0.025, expiry), paths,
                          precision=precision, seed=5, **kw)


def test_a_deals_gradients_are_the_average_of_its_slices():
    n, size = 16, 65536
    whole = _deal(n * size, 10.0)
    parts = [_deal(size, 10.0, path_offset=i * size) for i in range(n)]
    for k in FIELDS:
        mean = np.mean([getattr(p, k) for p in parts], axis=0)
        assert np.max(np.abs(getattr(whole, k) - mean)) <= 1e-10 * np.max(np.abs(mean))


def test_a_books_gradients_are_the_average_of_its_slices():
    m, pf = hjm.benchmark_market(), hjm.synthetic_portfolio(24, 5, seed=4)
    pf.periods = np.minimum(pf.periods, 10).astype(np.int32)

    def run(paths, first):
        print("[gpu] book Greeks: %d paths from %d" % (paths, first), flush=True)
        return hjm.portfolio_cva_greeks(m, pf, paths, horizon=5.0, precision=hjm.FP32_KAHAN, seed=5,
                                        path_offset=first)

    n, size = 8, 65536
    whole = run(n * size, 0)
    parts = [run(size, i * size) for i in range(n)]
    for k in FIELDS:
        mean = np.mean([getattr(p, k) for p in parts], axis=0)
        assert np.max(np.abs(getattr(whole, k) - mean)) <= 1e-10 * np.max(np.abs(mean))


@pytest.mark.parametrize("paths", [65536, 262144, 1048576])
def test_deals_of_many_paths_against_fp64(paths):
    a, b = _deal(paths, 10.0, hjm.FP64), _deal(paths, 10.0)
    for k in FIELDS:
        x, y = getattr(b, k), getattr(a, k)
        assert np.linalg.norm(x - y) <= 3e-6 * np.linalg.norm(y)


@pytest.mark.parametrize("paths,expiry", [(60001, 17.0), (600001, 1.5)])
def test_portions_do_not_change_the_sums(paths, expiry):
    a, b = _deal(paths, expiry), _deal(paths, expiry, regenerate_normals=True)
    assert a.stored_normals_bytes > 0 == b.stored_normals_bytes
    for k in FIELDS:
        assert np.array_equal(getattr(a, k), getattr(b, k))


def test_a_large_book_of_many_paths_against_fp64():
    # 65536 paths x 30y, 1024 swaps in 128 sets: the documented 1e-4 of the largest component
    m, pf = hjm.benchmark_market(), hjm.synthetic_portfolio(1024, 128, seed=7)

    def run(precision):
        print("[gpu] book Greeks: 65536 paths x 30y, precision %d" % precision, flush=True)
        return hjm.portfolio_cva_greeks(m, pf, 65536, horizon=30.0, precision=precision, seed=5)

    a, b = run(hjm.FP64), run(hjm.FP32_KAHAN)
    for k in FIELDS:
        x, y = getattr(b, k), getattr(a, k)
        assert np.max(np.abs(x - y)) <= 1e-4 * np.max(np.abs(y))
