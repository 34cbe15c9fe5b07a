"""The pruned float32 subsequence DTW scan: distances and indices are the
reference's exactly, whatever windows its bounds leave out.  Window counts
around 64 (the spread windows), 256 (a round of bounds) and the first rounds
without them, shapelets shorter than a bound's four terms, every kind of band, equal windows
(which overflow the candidate list) and data on which no bound prunes."""

import numpy as np
import pytest

import oracle
from wildboar_amd import distance as wd

pytestmark = pytest.mark.gpu


def _data(kind, n, t, lens, seed):
    rng = np.random.default_rng(seed)
    if kind == "integers":
        return (rng.integers(0, 3, (n, t)).astype(np.float64),
                [rng.integers(0, 3, L).astype(np.float64) for L in lens])
    if kind == "constant":
        X = np.full((n, t), 2.0)
        X[1:, t // 2:] = 0.5
        return X, [np.full(L, 1.0) for L in lens]
    if kind == "noise":  # the envelope covers nearly everything
        return rng.standard_normal((n, t)) * 0.01, [rng.standard_normal(L) * 5.0 for L in lens]
    X = rng.standard_normal((n, t)).cumsum(axis=1)
    S = [X[i % n, (t - L) // 2:][:L] + rng.standard_normal(L) * 0.1 for i, L in enumerate(lens)]
    return X, S


@pytest.mark.parametrize("kind", ["walks", "integers", "constant", "noise"])
@pytest.mark.parametrize("t,lens,r", [
    (40, (3, 5, 40, 37), 0.3),
    (83, (20, 20, 19, 21), 0.2),       # 63, 64 and 65 windows
    (300, (45, 46, 44), 0.1),          # 255, 256 and 257 windows
    (700, (64, 101, 128), 0.1),
    (900, (60, 128), 0.24),            # bands to 59 slots
    (600, (40, 33), 0.05),             # one-slot bands
    (400, (47, 50), 1.0),
    (1400, (60, 63), 0.1),             # on both sides of the fewest windows with bounds
    (5000, (30, 64), 0.2),             # several pauses between the bounds
])
def test_pruned_scan_is_exact(t, lens, r, kind):
    X, S = _data(kind, 4, t, lens, t + len(lens))
    for x in (X, X.astype(np.float32).astype(np.float64)):
        d, i = wd.pairwise_subsequence_distance(S, x, metric="dtw", metric_params={"r": r},
                                                return_index=True, precision="fp32")
        od, oi = oracle.subsequence(S, x, metric="dtw", r=r)
        np.testing.assert_array_equal(d, od)
        np.testing.assert_array_equal(i, oi)


@pytest.mark.parametrize("n,ns", [(1, 1), (7, 1), (8, 1), (9, 1), (65, 2), (2731, 3), (2732, 3),
                                  (3073, 3), (17000, 3)])
def test_candidates_of_many_tasks(n, ns):
    """A wave finishes the candidates of 8 tasks, of more from 8192 tasks on, of
    48 at most; integers leave from one to too many candidates a task."""
    rng = np.random.default_rng(n)
    X = rng.integers(0, 6, (n, 26)).astype(np.float64)
    X[::3] += rng.standard_normal((len(X[::3]), 26))
    S = [rng.integers(0, 6, 12).astype(np.float64) for _ in range(ns)]
    d, i = wd.pairwise_subsequence_distance(S, X, metric="dtw", metric_params={"r": 0.3},
                                            return_index=True, precision="fp32")
    od, oi = oracle.subsequence(S, X, metric="dtw", r=0.3)
    np.testing.assert_array_equal(np.asarray(d).reshape(od.shape), od)
    np.testing.assert_array_equal(np.asarray(i).reshape(oi.shape), oi)
