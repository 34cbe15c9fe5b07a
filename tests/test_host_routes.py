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


def _train_state_bytes(mode, nx, ny, t, band):
    m = _lib.WbxMetric(kind=_lib.DTW, precision=_lib.FP32, r=((band + 1) // 2 + 1e-6) / t)
    state, scratch = ctypes.c_int64(), ctypes.c_int64()
    _lib.check(_lib.load().wbx_dtw_train_sizes(ctypes.byref(m), mode, nx, ny, t, t,
                                               ctypes.byref(state), ctypes.byref(scratch)))
    return state.value


@pytest.mark.parametrize("n_pairs,t,band,few", [
    (4096, 256, 3, True), (8192, 256, 3, False), (8192, 256, 49, True), (12288, 256, 49, False),
    (12288, 256, 111, True), (16384, 256, 111, False), (2048, 1000, 9, True),
    (4096, 1000, 9, False), (8192, 1000, 111, True), (15808, 64, 9, True), (16448, 64, 49, False),
])
def test_few_pairs_form_of_training_by_band_and_length(n_pairs, t, band, few):
    """A wave for each pair's walk pays for fewer pairs the narrower the band
    and the longer the series.  The forms differ in the state they keep: a byte
    for two or four slots of a row, or two bits a slot in whole words."""
    up = lambda v: -(-v // 256) * 256
    planes = -(-n_pairs // 64) * 64 * t * 8 * -(-band // 32)
    bytes_2, bytes_4 = (up(n_pairs * t * -(-band // s)) for s in (2, 4))
    for mode, nx, ny in ((1, n_pairs, n_pairs), (0, n_pairs // 64, 64), (0, 1, n_pairs)):
        got = _train_state_bytes(mode, nx, ny, t, band) - up(4 * n_pairs)
        assert got in ((bytes_2, bytes_4) if few else (planes,))


def test_few_pairs_form_of_training_for_long_rows():
    """Sums over many columns of no multiple of 64 go one after the other in the
    other form."""
    up = lambda v: -(-v // 256) * 256
    for ny, few in ((10000, True), (9984, False), (16383, True), (16385, False)):
        got = _train_state_bytes(0, 1, ny, 256, 9) - up(4 * ny)
        assert (got == -(-ny // 64) * 64 * 256 * 8) == (not few)
