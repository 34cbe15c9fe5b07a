"""Calls too small to fill the chip take a group of lanes per pair with short
strips instead of a pair per lane.  The same pairs inside a call that fills it
take the lanes: both must agree bit for bit (float32: the same cells in the
same order; float64: the reference's arithmetic, also against the oracle).
Bands from 2 slots to the widest lane class, series shorter than the fill,
row counts around the groups of 8 steps, weights."""

import numpy as np
import pytest
import torch

import oracle
from wildboar_amd import _lib, device

pytestmark = pytest.mark.gpu

CASES = [  # tx, ty, r
    (5, 5, 0.4), (9, 9, 0.9), (16, 15, 0.2), (31, 31, 0.1), (64, 64, 0.1), (65, 61, 0.1),
    (71, 72, 0.2), (128, 128, 0.1), (150, 150, 0.1), (203, 203, 0.25), (129, 129, 0.8), (24, 24, 1.0), (43, 43, 0.52),
]


@pytest.mark.parametrize("metric", ["dtw", "wdtw"])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("tx,ty,r", CASES)
def test_small_call_equals_large_call(metric, precision, tx, ty, r):
    rng = np.random.default_rng(tx + ty)
    X = rng.standard_normal((3, tx)).cumsum(axis=1)
    Y = rng.standard_normal((7, ty)).cumsum(axis=1)
    dt = torch.float32 if precision == "fp32" else torch.float64
    Xd, Yd = torch.from_numpy(X).to("cuda", dt), torch.from_numpy(Y).to("cuda", dt)
    kw = dict(metric=metric, r=r, g=0.05, precision=precision)
    small = device.pairwise(Xd, Yd, **kw).cpu().numpy()
    one = device.pairwise(Xd[1:2], Yd[2:3], **kw).cpu().numpy()
    large = device.pairwise(Xd.repeat(400, 1), Yd.repeat(20, 1), **kw)[:3, :7].cpu().numpy()
    np.testing.assert_array_equal(small, large)
    np.testing.assert_array_equal(one[0, 0], small[1, 2])
    if precision == "fp64":
        np.testing.assert_array_equal(small, oracle.pairwise(X, Y, metric=metric, r=r, g=0.05))


@pytest.mark.parametrize("n", [2, 3, 40])
def test_small_singleton_and_paired(n):
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 90)).cumsum(axis=1)
    Y = rng.standard_normal((n, 90)).cumsum(axis=1)
    Xd, Yd = torch.from_numpy(X).cuda(), torch.from_numpy(Y).cuda()
    got = device.pairwise(Xd, metric="dtw", r=0.1, precision="fp64").cpu().numpy()
    full = oracle.pairwise(X, X, metric="dtw", r=0.1)
    want = np.triu(full, 1)
    np.testing.assert_array_equal(got, want + want.T)
    p = device.paired(Xd, Yd, metric="dtw", r=0.1, precision="fp64").cpu().numpy()
    np.testing.assert_array_equal(p, np.diag(oracle.pairwise(Y, X, metric="dtw", r=0.1)))


@pytest.mark.parametrize("metric", ["dtw", "euclidean"])
def test_output_in_the_memory_of_an_input(metric):
    # the distances then wait until every pair has read its series
    rng = np.random.default_rng(5)
    X = rng.standard_normal((300, 64)).cumsum(axis=1)
    Y = rng.standard_normal((64, 64)).cumsum(axis=1)
    Xd, Yd = torch.from_numpy(X).cuda(), torch.from_numpy(Y).cuda()
    want = device.pairwise(Xd, Yd, metric=metric, r=0.1, precision="fp64").clone()
    got = device.pairwise(Xd, Yd, metric=metric, r=0.1, precision="fp64", out=Xd)
    assert got.data_ptr() == Xd.data_ptr() and torch.equal(got, want)
    Sd = Yd.clone()
    want = device.pairwise(Sd, metric=metric, r=0.1, precision="fp64").clone()
    assert torch.equal(device.pairwise(Sd, metric=metric, r=0.1, precision="fp64", out=Sd), want)
    Pd = torch.from_numpy(X).cuda()
    want = device.paired(Pd, Pd.flip(0), metric=metric, r=0.1, precision="fp64").clone()
    flat = Pd.view(-1)[:300]
    assert torch.equal(device.paired(Pd, Pd.flip(0), metric=metric, r=0.1, precision="fp64",
                                     out=flat), want)


@pytest.mark.parametrize("nx,ny,kind", [(100, 200, 6), (300, 300, 2), (400, 320, 2)])
def test_two_waves_per_simd_take_the_lanes(nx, ny, kind):
    """B = 49: the lanes (kind 2) from a second wave per SIMD on, where they
    take 265 us on 90000 pairs of 800 and the group kernel (6) 307."""
    X = torch.randn((nx, 256), device="cuda")
    Y = torch.randn((ny, 256), device="cuda")
    _lib.prof_enable(True)
    try:
        device.pairwise(X, Y, metric="dtw", r=0.1, precision="fp32")
        _, launches, last = _lib.prof_take()
    finally:
        _lib.prof_enable(False)
    assert (launches, last) == (1, kind)
