"""CPU: the launch shapes of the run-time-schedule kernels.  Every length a
workgroup takes has one that the hardware holds, whatever the view: rows on both
sides, a length-fastest side, rows along X; one column, few and very many."""
import ctypes

import pytest

import p3dfft_amd

LDS = 160 * 1024
MAX_LEN = 8192
COUNTS = (1, 700, 3000, 100000)


def shapes(precision, form, tile, seg):
    L = p3dfft_amd.load(precision)
    s, t, b, o = ctypes.c_int(), ctypes.c_int(), ctypes.c_size_t(), ctypes.c_int()
    for n in range(1, MAX_LEN + 1):
        for c in COUNTS:
            assert L.p3dfft_amd_run_time_tile(n, form, c, tile, seg, ctypes.byref(s), ctypes.byref(t),
                                              ctypes.byref(b), ctypes.byref(o)) == 0
            yield n, c, s.value, t.value, b.value


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("tile,seg", [(0, 128), (32768, 64), (131072, 256)])
@pytest.mark.parametrize("form", [0, 1, 2])
def test_every_length_fits_the_lds(precision, form, tile, seg):
    bad = [(n, c, b) for n, c, s, t, b in shapes(precision, form, tile, seg) if b > LDS or s < 1]
    assert not bad, (len(bad), bad[:10])


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("tile,seg", [(0, 128), (131072, 256)])
@pytest.mark.parametrize("form", [0, 1, 2])
def test_every_length_has_threads(precision, form, tile, seg):
    """A prime stage holds its outputs in the registers of at most 1024 threads."""
    bad = [(n, c, s) for n, c, s, t, b in shapes(precision, form, tile, seg) if not (0 < t <= 1024 and t % 64 == 0)]
    assert not bad, (len(bad), bad[:10])


@pytest.mark.parametrize("precision", [8, 4])
def test_wide_offsets_reach_the_run_time_kernels(precision):
    """64-bit offsets above 4 GiB, and everywhere under the switch that the tests
    of that form use."""
    L = p3dfft_amd.load(precision)
    s, t, b, o = ctypes.c_int(), ctypes.c_int(), ctypes.c_size_t(), ctypes.c_int()

    def width(n, count):
        assert L.p3dfft_amd_run_time_tile(n, 0, count, 65536, 128, ctypes.byref(s), ctypes.byref(t), ctypes.byref(b),
                                          ctypes.byref(o)) == 0
        return o.value
    try:
        assert width(300, 1000) == 4
        assert width(1000, 1000 * 1000) == 8
        L.p3dfft_amd_set_wide_offsets(1)
        assert width(300, 1000) == 8
    finally:
        L.p3dfft_amd_set_wide_offsets(0)


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("form", [0, 2])
def test_plan_tile_sizes_reach_the_kernels(precision, form):
    """The tile sizes that a measured setup times are different tiles."""
    L = p3dfft_amd.load(precision)
    t, b, o = ctypes.c_int(), ctypes.c_size_t(), ctypes.c_int()
    got = []
    for tile in (32768, 65536, 131072):
        s = ctypes.c_int()
        assert L.p3dfft_amd_run_time_tile(500, form, 1000000, tile, 256, ctypes.byref(s), ctypes.byref(t),
                                          ctypes.byref(b), ctypes.byref(o)) == 0
        got.append(s.value)
    assert got[0] < got[1] < got[2], got


@pytest.mark.parametrize("n,like", [(3773, 3780), (1859, 1875), (946, 960)])
def test_11_and_13_points_are_register_stages(n, like):
    """They take as many FP32 columns as a length of small factors, and are not
    held back by what a prime stage over LDS can hold."""
    L = p3dfft_amd.load(4)
    s, t, b, o = ctypes.c_int(), ctypes.c_int(), ctypes.c_size_t(), ctypes.c_int()
    got = []
    for m in (n, like):
        assert L.p3dfft_amd_run_time_tile(m, 0, 100000, 131072, 256, ctypes.byref(s), ctypes.byref(t),
                                          ctypes.byref(b), ctypes.byref(o)) == 0
        got.append(s.value)
    assert got[0] == got[1], got


@pytest.mark.parametrize("precision", [8, 4])
def test_short_rows_fill_a_tile(precision):
    """Many short rows along X: a tile holds 256 values and more, and its row pairs
    divide every workgroup."""
    L = p3dfft_amd.load(precision)
    s, t, b, o = ctypes.c_int(), ctypes.c_int(), ctypes.c_size_t(), ctypes.c_int()
    for n in range(4, 40):
        assert L.p3dfft_amd_run_time_tile(n, 2, 1000000, 0, 128, ctypes.byref(s), ctypes.byref(t), ctypes.byref(b),
                                          ctypes.byref(o)) == 0
        assert s.value * n >= 256 and t.value % s.value == 0, (n, s.value, t.value)


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("form", [3, 4])
def test_copies_have_loads_in_flight(precision, form):
    """Op 'n': at most four values a thread, up to the largest workgroup."""
    for n, c, s, t, b in shapes(precision, form, 0, 128):
        assert 0 < b <= LDS and t % 64 == 0 and t <= 1024, (n, c, s, t, b)
        assert t == 1024 or 4 * t >= n * s, (n, c, s, t)


@pytest.mark.parametrize("precision", [8, 4])
def test_other_lengths_are_refused(precision):
    L = p3dfft_amd.load(precision)
    s, t, b, o = ctypes.c_int(), ctypes.c_int(), ctypes.c_size_t(), ctypes.c_int()
    for n in (0, MAX_LEN + 1):
        assert L.p3dfft_amd_run_time_tile(n, 0, 1, 65536, 128, ctypes.byref(s), ctypes.byref(t), ctypes.byref(b),
                                          ctypes.byref(o)) == -1
    L.p3dfft_amd_clear_error()
