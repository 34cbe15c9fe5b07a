"""The pruned scaled DTW search (calls with enough series and patterns) against
the exhaustive windows of the same tasks (calls too small for it) and against
the oracle: bit-identical distances and indices.  Window counts below, at and
just past 64 and its multiples, every register class of the band, repeated
values (equal windows), patterns planted in the series and flat windows."""

import numpy as np
import pytest

import oracle
from wildboar_amd import distance as wd

pytestmark = pytest.mark.gpu


def _data(kind, n, t, lens, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((n, t)).cumsum(axis=1)
    S = [rng.standard_normal(L).cumsum() for L in lens]
    if kind == "integers":
        X = rng.integers(0, 4, (n, t)).astype(np.float64)
        S = [rng.integers(0, 4, L).astype(np.float64) for L in lens]
    elif kind == "planted":
        for i in range(n):
            s = S[i % len(S)]
            o = int(rng.integers(0, t - len(s) + 1))
            X[i, o:o + len(s)] = 3.0 * s + rng.standard_normal(len(s)) * 0.05
    elif kind == "copies":  # distances of rounding size: settled by the exact pass
        for i in range(n):
            s = S[i % len(S)]
            for o in range(0, t - len(s) + 1, len(s) + 3):
                X[i, o:o + len(s)] = s * (1.0 + o) + i
    elif kind == "sine":  # every period again, up to rounding
        X = np.sin(np.arange(t) * (2 * np.pi / 25) + rng.uniform(0, 6, (n, 1)))
        S = [np.sin(np.arange(L) * (2 * np.pi / 25) + rng.uniform(0, 6)) for L in lens]
    elif kind == "flat":
        X[:, t // 3: t // 3 + min(40, t // 2)] = 1.5
    return X, S


CASES = [  # t, lengths, r
    (40, (3, 5, 8, 12), 0.2),
    (75, (12, 12, 12), 0.1),       # 64 windows
    (76, (12, 12), 0.1),           # 65 windows
    (139, (12, 12, 11), 0.3),      # 128 and 129 windows
    (300, (30, 64, 101), 0.1),
    (260, (40, 90), 0.3),          # bands 25 and 55
    (200, (3, 4, 6), 1.0),
]


@pytest.mark.parametrize("kind", ["walks", "integers", "planted", "copies", "flat",
                                  "sine"])
@pytest.mark.parametrize("t,lens,r", CASES)
def test_pruned_search_equals_every_window(t, lens, r, kind):
    n = 6
    X, S = _data(kind, n, t, lens, t)
    call = lambda x: wd.pairwise_subsequence_distance(
        S, x, metric="dtw", metric_params={"r": r}, scale=True, return_index=True)
    small_d, small_i = call(X)
    # as many series as give the search its tasks in every class of the call
    reps = -(-1100 // n)
    large_d, large_i = call(np.tile(X, (reps, 1)))
    for k in range(reps):
        np.testing.assert_array_equal(large_d[k * n:(k + 1) * n], small_d)
        np.testing.assert_array_equal(large_i[k * n:(k + 1) * n], small_i)
    od, oi = oracle.scaled_subsequence(S, X, metric="dtw", r=r)
    np.testing.assert_array_equal(small_d, od)
    np.testing.assert_array_equal(small_i, oi)
