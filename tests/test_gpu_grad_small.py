"""Differentiable DTW of few pairs (several lanes per pair, the path walked on
the scalar unit) against the pair-per-lane form: the same cells, decisions and
gradient arithmetic, so a pair's distance and gradients are the same bits
whichever form its call takes.  Bands of 1 slot to the widest of the form, on
both sides of its 32-slot decision words, unequal lengths, tied integer data,
identical series (D = 0)."""

import numpy as np
import pytest
import torch

from wildboar_amd.dtw import dtw, paired_dtw

pytestmark = pytest.mark.gpu

LARGE = 16384 + 64  # pairs: past the small form

CASES = [  # tx, ty, r
    (1, 1, 1.0), (6, 6, 0.0), (9, 7, 0.3), (40, 40, 0.1), (33, 41, 0.2), (41, 33, 0.2),
    (160, 160, 0.1), (165, 165, 0.1), (170, 170, 0.1), (256, 256, 0.1), (300, 310, 0.17),
    (257, 257, 0.218),
]


def _grads(fn, X, Y, G, r):
    X, Y = X.clone().requires_grad_(True), Y.clone().requires_grad_(True)
    D = fn(X, Y, r)
    gx, gy = torch.autograd.grad((D * G).sum(), (X, Y))
    return D.detach(), gx, gy


@pytest.mark.parametrize("data", ["walks", "integers"])
@pytest.mark.parametrize("tx,ty,r", CASES)
def test_small_form_equals_lane_form(tx, ty, r, data):
    rng = np.random.default_rng(tx * 7 + ty)
    n = 37

    def series(t):
        if data == "integers":
            return rng.integers(-2, 3, (n, t))
        return rng.standard_normal((n, t)).cumsum(axis=1)

    X = torch.from_numpy(series(tx).astype(np.float32)).cuda()
    Y = torch.from_numpy(series(ty).astype(np.float32)).cuda()
    if tx == ty:
        Y[3] = X[3]
    G = torch.from_numpy(rng.standard_normal(n)).cuda()
    small = _grads(paired_dtw, X, Y, G, r)
    reps = -(-LARGE // n)
    large = _grads(paired_dtw, X.repeat(reps, 1), Y.repeat(reps, 1), G.repeat(reps), r)
    for s, l in zip(small, large):
        assert torch.equal(s, l[:n])


@pytest.mark.parametrize("nx,ny", [(1, 1), (1, 5), (5, 1), (3, 64), (2, 130), (300, 3)])
def test_small_matrix_sums_pairs(nx, ny):
    rng = np.random.default_rng(nx + ny)
    X = torch.from_numpy(rng.standard_normal((nx, 70)).cumsum(axis=1).astype(np.float32)).cuda()
    Y = torch.from_numpy(rng.standard_normal((ny, 66)).cumsum(axis=1).astype(np.float32)).cuda()
    G = torch.from_numpy(rng.standard_normal((nx, ny))).cuda()
    D, gx, gy = _grads(dtw, X, Y, G, 0.2)
    pd, px, py = _grads(paired_dtw, X.repeat_interleave(ny, 0), Y.repeat(nx, 1), G.reshape(-1),
                        0.2)
    assert torch.equal(D, pd.reshape(nx, ny))
    px, py = px.double().reshape(nx, ny, -1), py.double().reshape(nx, ny, -1)
    # a float32 sum of m terms is within m u of the sum of their magnitudes
    u = 2.0**-24
    assert ((gx.double() - px.sum(1)).abs() <= ny * u * px.abs().sum(1) + 1e-30).all()
    assert ((gy.double() - py.sum(0)).abs() <= nx * u * py.abs().sum(0) + 1e-30).all()
