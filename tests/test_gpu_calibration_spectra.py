"""PCA calibration where its eigensolver has special cases.

Too few days for three factors, equal leading eigenvalues, a covariance that is diagonal,
decoupled or zero, and more windows than are solved at a time. A solver that is backward
stable leaves residuals of n^2 = 51^2 roundings of the largest eigenvalue at most, 2.9e-13 of
it, whatever the gaps: eigenvalues against numpy's, C r = lambda r for each raw loading,
r_f . r_g = lambda_f or 0.
"""
import numpy as np
import pytest

import cva_hjm_cuda_amd as hjm

pytestmark = pytest.mark.gpu

N = 51


def _history(kind):
    rng = np.random.default_rng(5)
    q = np.linalg.qr(rng.standard_normal((N, N)))[0]
    if kind == "zero":
        d = np.zeros((8, N))
    elif kind == "one tenor":
        d = np.zeros((9, N))
        d[:, 7] = rng.standard_normal(9)
    elif kind == "diagonal, equal":
        d = np.repeat(np.eye(N)[[5, 9, 50]], 2, axis=0) * np.tile([1.0, -1.0], 3)[:, None]
    elif kind == "dense, equal":
        d = np.repeat(q[:4], 2, axis=0) * np.tile([1.0, -1.0], 4)[:, None]
    elif kind == "decoupled":
        d = rng.standard_normal((30, N))
        d[::2, 20:] = 0.0
        d[1::2, :20] = 0.0
    elif kind == "graded":
        d = rng.standard_normal((200, N)) * 10.0 ** -np.arange(N)[None, ::-1]
    else:
        d = rng.standard_normal((2, N)) if kind == "two days" else rng.standard_normal((64, N))
    scale = 1e150 if kind == "huge" else 1e-3
    return scale * np.concatenate([np.zeros((1, N)), np.cumsum(d, axis=0)])


def _check(curves, ev, raw):
    c = np.cov(np.diff(curves, axis=0), rowvar=False) * 252.0
    s = max(np.max(np.abs(c)), 1e-300)
    c, ev, raw = c / s, ev / s, raw.reshape(3, N) / np.sqrt(s)
    want = np.sort(np.linalg.eigvalsh(c))[::-1]
    tol = 2.0 * N * N * 2.0 ** -53 * max(want[0], 1e-300)
    assert np.max(np.abs(ev - want)) <= tol
    lam = np.maximum(ev[:3], 0.0)
    assert np.max(np.abs(raw @ raw.T - np.diag(lam))) <= tol
    assert np.max(np.abs(raw @ c - lam[:, None] * raw)) <= tol * np.sqrt(max(want[0], 1e-300))


@pytest.mark.parametrize("kind", ["zero", "one tenor", "diagonal, equal", "dense, equal", "decoupled",
                                  "graded", "two days", "full", "huge"])
def test_spectra(kind):
    print("[gpu] calibration, %s" % kind, flush=True)
    curves = _history(kind)
    g = hjm.calibrate_pca(curves)
    _check(curves, g.eigenvalues[0], g.raw_loadings[0])


def test_more_windows_than_a_batch():
    print("[gpu] calibration, 4099 windows of 7 curves", flush=True)
    rng = np.random.default_rng(6)
    curves = 1e-3 * np.cumsum(rng.standard_normal((4105, N)), axis=0)
    g = hjm.calibrate_pca(curves, window=7, nwindows=4099)
    for w in (0, 1, 4095, 4096, 4098):
        _check(curves[w:w + 7], g.eigenvalues[w], g.raw_loadings[w])
