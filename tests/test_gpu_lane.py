"""The exact-band float32 lane kernels with a shared x series per wave (matrix
rows cut into waves of 64 columns), with and without weights in SGPRs, against the group kernel, which computes
the same cells in the same order: bit-identical.  Column counts on both sides
of whole waves, series shorter than a group of rows, remainders of 8 rows,
unequal lengths, the narrowest and widest bands; and against the oracle."""

import numpy as np
import pytest

import oracle
from wildboar_amd import _lib
from wildboar_amd import distance as wd

pytestmark = pytest.mark.gpu

CASES = [  # nx, ny, tx, ty, r -> band
    (3, 64, 45, 45, 0.12),    # B = 9
    (2, 128, 7, 7, 0.9),      # B = 11, fewer rows than a group
    (3, 63, 131, 131, 0.1),   # B = 25, last wave partly idle
    (5, 65, 131, 131, 0.1),   # x per lane: a second wave per row would idle
    (2, 64, 98, 100, 0.1),    # unequal, B = 19
    (2, 64, 100, 98, 0.1),
    (3, 192, 256, 256, 0.1),  # B = 49
    (2, 64, 300, 300, 0.17),  # B = 101
    (2, 64, 301, 301, 0.187), # B = 111
    (1, 64, 8, 8, 0.7),
]


@pytest.mark.parametrize("metric", ["dtw", "wdtw"])
@pytest.mark.parametrize("nx,ny,tx,ty,r", CASES)
def test_shared_x_waves_match_group_kernel(nx, ny, tx, ty, r, metric):
    rng = np.random.default_rng(nx * ny + tx)
    X = rng.standard_normal((nx, tx)).cumsum(axis=1)
    Y = rng.standard_normal((ny, ty)).cumsum(axis=1)
    # many rows of x, so that the matrix fills the chip and the lanes run it
    reps = -(-140000 // (nx * ny))
    X = np.tile(X, (reps, 1))
    params = {"r": r} if metric == "dtw" else {"r": r, "g": 0.1}
    call = lambda: wd.pairwise_distance(X, Y, metric=metric, metric_params=params,
                                        precision="fp32")
    got = call()
    _lib.set_policy(2)
    try:
        want = call()
    finally:
        _lib.set_policy(0)
    np.testing.assert_array_equal(got, want)
    ref = oracle.pairwise(X[:nx], Y, metric=metric, r=r, g=0.1)
    # (1 + u)^(lx + ly) and the rounding of the inputs
    tol = (tx + ty + 8) * 2.0**-24 * (1 + np.abs(X).max() ** 2)
    np.testing.assert_allclose(got[:nx], ref, rtol=1e-5, atol=tol)


@pytest.mark.parametrize("metric", ["ddtw", "wddtw"])
@pytest.mark.parametrize("t,r", [(7, 1.0), (8, 0.9), (15, 1.0), (22, 0.97), (23, 1.0), (30, 0.99),
                                 (50, 1.0), (57, 0.97), (57, 0.99)])
def test_slopes_under_a_wider_band(t, r, metric):
    """Slopes are two values shorter than their series and keep its band, which
    may be wider than they are long: slots without a weight."""
    rng = np.random.default_rng(t)
    X = rng.standard_normal((3, t)).cumsum(axis=1)
    Y = rng.standard_normal((130, t)).cumsum(axis=1)
    params = {"r": r} if metric == "ddtw" else {"r": r, "g": 0.1}
    big = np.tile(X, (400, 1))  # fills the chip: lanes
    call = lambda x: wd.pairwise_distance(x, Y, metric=metric, metric_params=params,
                                          precision="fp32")
    got = call(big)
    _lib.set_policy(2)
    try:
        want = call(big)
    finally:
        _lib.set_policy(0)
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(got[:3], call(X))  # few pairs: several lanes each
    ref = oracle.pairwise(X, Y, metric=metric, r=r, g=0.1)
    # slopes are rounded to float32 (|slope| <= 2 |x|), then (1 + u)^(lx + ly)
    tol = (2 * t + 8) * 2.0**-24 * (1 + 4 * np.abs(X).max() ** 2)
    np.testing.assert_allclose(got[:3], ref, rtol=1e-5, atol=tol)
