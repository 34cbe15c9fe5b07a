"""Differentiable DTW of x series that are not finite everywhere.  The distance
is then not finite and the gradient 0 or NaN: NaN at the values themselves and
at columns of y that the band can match to them, 0 elsewhere.  The finite pairs
of the call do not change."""

import numpy as np
import pytest
import torch

from wildboar_amd.dtw import dtw, paired_dtw

pytestmark = pytest.mark.gpu

T, R = 24, 0.2
W = 4  # floor(T R): |i - j| < W


def _series(n, seed):
    return np.random.default_rng(seed).standard_normal((n, T)).astype(np.float32)


def _grads(fn, X, Y):
    X = torch.from_numpy(X).cuda().requires_grad_(True)
    Y = torch.from_numpy(Y).cuda().requires_grad_(True)
    D = fn(X, Y, R)
    gx, gy = torch.autograd.grad(D.sum(), (X, Y))
    return [v.detach().cpu().numpy() for v in (D, gx, gy)]


@pytest.mark.parametrize("bad", [np.nan, -np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("n", [40, 20000])  # the few-pairs form and a pair per lane
def test_paired(n, bad):
    X, Y = _series(n, 1), _series(n, 2)
    clean = _grads(paired_dtw, X, Y)
    rows = {3: 0, 9: 7, 17: 12, 31: T - 1}
    for p, i in rows.items():
        X[p, i] = bad
    D, gx, gy = _grads(paired_dtw, X, Y)
    ok = np.ones(n, bool)
    for p, i in rows.items():
        ok[p] = False
        np.testing.assert_array_equal(np.isnan(gx[p]), ~np.isfinite(X[p]))
        near = np.abs(np.arange(T) - i) < W
        assert np.isnan(gy[p][near]).any() and not np.isnan(gy[p][~near]).any()
        assert (np.nan_to_num(gx[p]) == 0).all() and (np.nan_to_num(gy[p]) == 0).all()
    for got, want in zip((D, gx, gy), clean):
        np.testing.assert_array_equal(got[ok], want[ok])


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("nx,ny", [(3, 64), (300, 64), (3090, 64), (300, 70)])
def test_matrix(nx, ny, bad):
    X, Y = _series(nx, 3), _series(ny, 4)
    X[1, 10] = bad
    D, gx, gy = _grads(dtw, X, Y)
    assert not np.isfinite(D[1]).any() and np.isfinite(np.delete(D, 1, 0)).all()
    np.testing.assert_array_equal(np.isnan(gx), ~np.isfinite(X))
    near = np.abs(np.arange(T) - 10) < W
    assert np.isnan(gy[:, near]).any(1).all() and not np.isnan(gy[:, ~near]).any()
