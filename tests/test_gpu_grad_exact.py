"""Differentiable DTW on exact-band lanes, with x from SGPRs (grids of whole
waves) and from VGPRs (lists of pairs): bands on both sides of the 32-slot
decision words and the narrowest and widest exact ones.  D is homogeneous of
degree 1 in (x, y) jointly, so <dD/dx, x> + <dD/dy, y> = D, which holds only
when the walked path has the cost the recurrence found.  Grids of one and of
several waves per x series and of waves across series."""

import numpy as np
import pytest
import torch

from wildboar_amd.dtw import dtw, paired_dtw

pytestmark = pytest.mark.gpu


def _grads(fn, X, Y, G, r):
    X, Y = X.clone().requires_grad_(True), Y.clone().requires_grad_(True)
    D = fn(X, Y, r)
    gx, gy = torch.autograd.grad((D * G).sum(), (X, Y))
    return D.detach(), gx, gy


@pytest.mark.parametrize("data", ["walks", "integers"])
@pytest.mark.parametrize("nx,ny", [(260, 64), (130, 128), (237, 70)])  # more than few pairs
@pytest.mark.parametrize("slots", [9, 31, 33, 49, 63, 65, 97, 111])
def test_exact_forms(slots, nx, ny, data):
    rng = np.random.default_rng(slots)
    t = 131
    r = (slots - 1) / 2 / t + 1e-6

    def series(n):
        if data == "integers":
            return rng.integers(-2, 3, (n, t))
        return rng.standard_normal((n, t)).cumsum(axis=1)

    X = torch.from_numpy(series(nx).astype(np.float32)).cuda()
    Y = torch.from_numpy(series(ny).astype(np.float32)).cuda()
    G = torch.from_numpy(rng.uniform(0.5, 2.0, (nx, ny))).cuda()
    D, gx, gy = _grads(dtw, X, Y, G, r)
    Xp, Yp, Gp = X.repeat_interleave(ny, 0), Y.repeat(nx, 1), G.reshape(-1)
    Dp, px, py = _grads(paired_dtw, Xp, Yp, Gp, r)
    assert torch.equal(D.reshape(-1), Dp)

    # sums of m float32 terms are within m u of the sum of their magnitudes
    u = 2.0**-24
    qx, qy = px.double().reshape(nx, ny, t), py.double().reshape(nx, ny, t)
    assert ((gx.double() - qx.sum(1)).abs() <= ny * u * qx.abs().sum(1) + 1e-30).all()
    assert ((gy.double() - qy.sum(0)).abs() <= nx * u * qy.abs().sum(0) + 1e-30).all()

    # a path has at most 2 t cells; each adds terms of at most G/D |x|max (|x| +
    # |y|)max to the products, rounded a few times in sums of at most t terms;
    # D^2 is a float32 sum of at most 2 t squares
    pos = Dp > 0
    hom = (px.double() * Xp.double()).sum(1) + (py.double() * Yp.double()).sum(1)
    big = torch.maximum(Xp.abs().amax(1), Yp.abs().amax(1)).double()
    bound = 2 * t * u * (Gp * Dp + 2 * t * Gp / Dp.clamp(min=1e-30) * 4 * big**2)
    assert ((hom - Gp * Dp).abs() <= bound)[pos].all()


@pytest.mark.parametrize("nx,ny,t,r", [
    (3073, 64, 20, 0.1),   # 385 blocks of 8 series, the last with one; band 5 (padded to 8)
    (1540, 128, 45, 0.45), # two waves per x series, band 41
    (2048, 64, 66, 0.7),   # a wide band (93 slots) at its own smallest count
    (2048, 64, 110, 0.47), # bands of 101 and 111 slots: the most shared memory
    (2055, 64, 120, 0.4675),
    (3080, 64, (30, 41), 0.2),
])
def test_shared_prefix_blocks(nx, ny, t, r):
    """Full-chip grids (eight x series share a block's window of y prefix sums)
    against the same rows in calls too small for it: the same terms."""
    tx, ty = t if isinstance(t, tuple) else (t, t)
    rng = np.random.default_rng(tx)
    X = torch.from_numpy(rng.standard_normal((nx, tx)).cumsum(axis=1).astype(np.float32)).cuda()
    Y = torch.from_numpy(rng.standard_normal((ny, ty)).cumsum(axis=1).astype(np.float32)).cuda()
    G = torch.from_numpy(rng.uniform(0.5, 2.0, (nx, ny))).cuda()
    D, gx, gy = _grads(dtw, X, Y, G, r)
    sy = torch.zeros_like(gy, dtype=torch.float64)
    for i in np.array_split(np.arange(nx), nx * ny // 17000):  # past the few-pairs form
        i = slice(i[0], i[-1] + 1)
        d, px, py = _grads(dtw, X[i], Y, G[i], r)
        assert torch.equal(D[i], d)
        assert torch.equal(gx[i], px)  # one order of sums over the row's pairs
        sy += py.double()
    # two float32 sums of nx terms in different orders
    _, _, py = _grads(paired_dtw, X.repeat_interleave(ny, 0), Y.repeat(nx, 1), G.reshape(-1), r)
    mag = py.double().abs().reshape(nx, ny, ty).sum(0)
    u = 2.0**-24
    assert ((gy.double() - sy).abs() <= 2 * nx * u * mag + 1e-30).all()
