"""Certified float32 argmin: the wave-per-row candidate selection and the heap
replay over its lists, at the edges of their 64- and 256-column groups, the
64-word batches of the candidate bits (4096 columns) and the heap sizes, with
tied and equal distances.  Float32 requests return the reference's indices,
order and float64 distances exactly, so every comparison is exact."""

import numpy as np
import pytest

import oracle
from wildboar_amd import distance as wd

pytestmark = pytest.mark.gpu


def _series(n, t, seed, kind):
    rng = np.random.default_rng(seed)
    if kind == "integers":  # few distinct distances
        return rng.integers(0, 3, (n, t)).astype(np.float64)
    if kind == "equal":  # every column is a candidate
        return np.tile(rng.standard_normal(t), (n, 1))
    return rng.standard_normal((n, t)).cumsum(axis=1)


@pytest.mark.parametrize("kind", ["walks", "integers", "equal"])
@pytest.mark.parametrize("ny,k", [(1, 1), (3, 3), (63, 1), (64, 5), (65, 32), (255, 5), (257, 1),
                                  (4096, 5), (4097, 3), (8200, 1)])
def test_certified_argmin_edges(kind, ny, k):
    nx, t = 5, 12
    X, Y = _series(nx, t, 1, kind), _series(ny, t, 2, kind)
    for metric in ("dtw", "euclidean"):
        params = {} if metric == "euclidean" else {"r": 0.2}
        idx, dist = wd.argmin_distance(X, Y, k=k, metric=metric, metric_params=params,
                                       return_distance=True, precision="fp32")
        oi, od = oracle.argmin(X, Y, k=k, metric=metric, r=0.2)
        np.testing.assert_array_equal(idx, oi)
        np.testing.assert_array_equal(dist, od)


@pytest.mark.parametrize("k", [64, 65])
def test_replay_heap_in_lds_and_in_memory(k):
    X, Y = _series(4, 20, 3, "walks"), _series(300, 20, 4, "walks")
    idx, dist = wd.argmin_distance(X, Y, k=k, metric="dtw", metric_params={"r": 0.1},
                                   return_distance=True)
    oi, od = oracle.argmin(X, Y, k=k, metric="dtw", r=0.1)
    np.testing.assert_array_equal(idx, oi)
    np.testing.assert_array_equal(dist, od)


@pytest.mark.parametrize("nx,ny,k", [(4096, 3, 1), (4097, 66, 5), (8193, 70, 3), (266300, 3, 2)])
def test_many_rows(nx, ny, k):
    """From 4097 rows on a wave takes several, 64 at most."""
    X, Y = _series(nx, 12, 5, "walks"), _series(ny, 12, 6, "walks")
    X[::5] = Y[0]  # some rows with a distance of 0
    idx, dist = wd.argmin_distance(X, Y, k=k, metric="dtw", metric_params={"r": 0.2},
                                   return_distance=True, precision="fp32")
    oi, od = oracle.argmin(X, Y, k=k, metric="dtw", r=0.2)
    np.testing.assert_array_equal(idx, oi)
    np.testing.assert_array_equal(dist, od)
