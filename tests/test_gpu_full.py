"""The full-matrix kernel (r = 1) at every number of columns per lane that its
plan takes from the size of the call: a matrix inside a large call against the
same pairs in small ones (float32: the same cells, bit for bit) and, in
float64, against the oracle.  Lengths around multiples of the columns per
lane, fewer rows than lanes, rows around the groups of 4 and 8 steps."""

import numpy as np
import pytest
import torch

import oracle
from wildboar_amd import device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("tx,ty", [(1, 1), (2, 9), (9, 2), (7, 100), (100, 100), (101, 128),
                                   (64, 255), (275, 275), (300, 276), (37, 512), (512, 37)])
def test_full_matrix_small_and_large_calls(tx, ty, precision):
    rng = np.random.default_rng(tx + 3 * ty)
    X = rng.standard_normal((3, tx)).cumsum(axis=1)
    Y = rng.standard_normal((5, ty)).cumsum(axis=1)
    dt = torch.float32 if precision == "fp32" else torch.float64
    Xd, Yd = torch.from_numpy(X).to("cuda", dt), torch.from_numpy(Y).to("cuda", dt)
    kw = dict(metric="dtw", r=1.0, precision=precision)
    small = device.pairwise(Xd, Yd, **kw).cpu().numpy()
    for reps in (20, 300, 1600):
        got = device.pairwise(Xd.repeat(reps, 1), Yd.repeat(7, 1), **kw)
        np.testing.assert_array_equal(got[-3:, -5:].cpu().numpy(), small)
    if precision == "fp64":
        np.testing.assert_array_equal(small, oracle.pairwise(X, Y, metric="dtw", r=1.0))
