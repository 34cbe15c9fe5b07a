"""Rules of the dispatch that decide on the host, called in the built library:
no GPU needed."""

import ctypes

import pytest

from wildboar_amd import _lib

_GRID = 0


class _PairSpec(ctypes.Structure):
    _fields_ = [("mode", ctypes.c_int), ("n_pairs", ctypes.c_int64), ("ny", ctypes.c_int64),
                ("pa", ctypes.c_void_p), ("pb", ctypes.c_void_p), ("out", ctypes.c_void_p),
                ("ld", ctypes.c_int64)]


def _exact_w_waves(nx, ny, lx, ly, band):
    fn = _lib.load()._ZN3wbx18lane_exact_w_wavesERKNS_8PairSpecEiii
    fn.restype = ctypes.c_int64
    return fn(ctypes.byref(_PairSpec(_GRID, nx * ny, ny)), lx, ly, band)


@pytest.mark.parametrize("t", [6, 7, 20, 33, 50, 57])
def test_weighted_lanes_need_a_weight_for_every_slot(t):
    """Slopes of series of t values are t - 2 long and have t - 2 weights, but
    keep the band width w of the series, up to t: the kernel that reads w
    weights serves w <= t - 2 only."""
    n = t - 2
    for w in range(5, t + 1):
        waves = _exact_w_waves(1000, 1000, n, n, 2 * w - 1)
        assert waves == (16000 if w <= n and 2 * w - 1 <= 111 else 0), w
