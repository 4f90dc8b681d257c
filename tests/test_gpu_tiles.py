"""Run-time-schedule column passes whose tile is near what a workgroup holds: the
widest tile fills the LDS without room for the skew of its blocks, or a prime
stage fills the registers, with enough columns for whole row segments, and the
Chebyshev axis whose extension has such a length.  Against the FP64 oracle, tolerances as test_gpu_parity.py."""
import numpy as np
import pytest

from test_gpu_parity import TOL, cheby_tol, lib_setup, oplan, rel

pytestmark = pytest.mark.gpu


def check(precision, shape):
    nx, ny, nz = shape
    a = np.random.default_rng(ny + nz).standard_normal((nz, ny, nx))
    o = oplan(nx, ny, nz)
    ref = o.ftran_r2c(a, "fft")
    with lib_setup(precision, nx, ny, nz) as P:
        assert rel(P.ftran_r2c(a, "fft"), ref) < TOL[precision]
        assert rel(P.btran_c2r(ref, "tff"), o.btran_c2r(ref, "tff")[0]) < TOL[precision]


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", [1714, 2400, 2500, 5000])
def test_no_room_for_the_skew(precision, n):
    check(precision, (2, n, 1056))  # 2112 columns


@pytest.mark.parametrize("shape", [(2, 1881, 1056), (2, 1911, 1056), (6, 3762, 3), (6, 3, 3773), (2, 1, 7513)])
def test_prime_stage_registers(shape):
    """Prime stages of 11 and 13 just above what the threads of a workgroup hold
    at the widest tile of FP32"""
    check(4, shape)


@pytest.mark.parametrize("precision", [8, 4])
def test_no_room_for_the_skew_few_columns(precision):
    check(precision, (6, 4800, 3))
    check(precision, (6, 3, 5000))


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", [26, 169, 286, 2197])
def test_stages_of_11_and_13(precision, n):
    """In registers: alone, between factors, several in a row; decimation in time
    (rows) and in frequency (X c2r, length-fastest input), a row map."""
    for shape, cut, stride1 in (((n, 3, 4), None, False), ((4, n, 300), None, False), ((10, 7, n), None, True),
                                ((10, 6, n), 2 * (n // 3), True), ((10, n, 4), 2 * (n // 3), False)):
        nx, ny, nz = shape
        c = (None, None, cut) if stride1 else (None, cut, None)
        a = np.random.default_rng(n).standard_normal((nz, ny, nx))
        o = oplan(nx, ny, nz, *c, stride1=stride1)
        ref = o.ftran_r2c(a, "fft")
        with lib_setup(precision, nx, ny, nz, *c, stride1=stride1) as P:
            assert rel(P.ftran_r2c(a, "fft"), ref) < TOL[precision]
            assert rel(P.btran_c2r(ref, "tff"), o.btran_c2r(ref, "tff")[0]) < TOL[precision]


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", [187, 221, 266, 2431])
def test_stages_of_both_kinds(precision, n):
    """11 and 13 points in registers beside larger primes over LDS, and larger ones
    alone, along each axis"""
    for shape in ((n, 3, 4), (4, n, 300), (10, 7, n)):
        check(precision, shape)


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", range(1, 16))
def test_short_rows(precision, n):
    """Rows of one stage (up to 10 points) and just above along X, in wide tiles
    of which the last is partial and holds an odd row; pruned modes."""
    for ny, nz, cut in ((5, 7, None), (201, 331, None), (6, 9, 2 * ((n + 1) // 3))):
        if cut == 0:
            continue
        a = np.random.default_rng(n).standard_normal((nz, ny, n))
        o = oplan(n, ny, nz, cut)
        ref = o.ftran_r2c(a, "fft")
        with lib_setup(precision, n, ny, nz, cut) as P:
            assert rel(P.ftran_r2c(a, "fft"), ref) < TOL[precision]
            assert rel(P.btran_c2r(ref, "tff"), o.btran_c2r(ref, "tff")[0]) < TOL[precision]


@pytest.mark.parametrize("precision", [8, 4])
def test_chebyshev_extension(precision):
    """nz = 1251: the even extension has 2500 points"""
    nx, ny, nz = 2, 1056, 1251
    a = np.random.default_rng(5).standard_normal((nz, ny, nx))
    ref = oplan(nx, ny, nz).cheby(a, 2.0)
    with lib_setup(precision, nx, ny, nz) as P:
        assert rel(P.cheby(a, 2.0), ref) < cheby_tol(precision, nz, 2.0)


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("shape,cut", [((30, 50, 21), (None, None, None)), ((30, 50, 21), (20, 30, 15)),
                                       ((22, 77, 100), (None, 50, 64))])
def test_wide_offsets_with_maps(precision, shape, cut):
    """The 64-bit-offset form of the row-addressed kernel against the 32-bit
    one: plain rows, pruned rows, DCT-I and DST-I extensions.  Identical bits."""
    nx, ny, nz = shape
    a = np.random.default_rng(nz).standard_normal((nz, ny, nx))
    res = []
    for wide in (0, 1):
        with lib_setup(precision, nx, ny, nz, *cut, ow=False) as P:
            P.lib.p3dfft_amd_set_wide_offsets(wide)
            try:
                for z in "tcs":
                    s = P.ftran_r2c(a, "ff" + z)
                    res.append((s, P.btran_c2r(s, z + "ff")))
            finally:
                P.lib.p3dfft_amd_set_wide_offsets(0)
    for (s0, b0), (s1, b1) in zip(res[:3], res[3:]):
        assert np.array_equal(s0, s1) and np.array_equal(b0, b1)
