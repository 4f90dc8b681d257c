"""The run-time-schedule kernels (lengths without specialised kernels) at the
lengths where they can go wrong, against the FP64 oracle: one point, single
stages, the largest radix in registers, primes just above it, products of
large primes, prime stages first, in the middle and last, three and four
stages, and the longest lengths a tile holds; each as X, Y and Z axis, in both
layouts, with and without cuts.  Tolerances as test_gpu_parity.py."""
import numpy as np
import pytest

from test_gpu_parity import TOL, lib_setup, oplan, rel

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 7, 9, 10, 11, 14, 22, 25, 77, 97, 100, 121, 143, 210, 243, 250, 289, 300, 361, 441, 500, 630, 1000]
LONG = [1331, 2310, 3000, 4099, 6561, 8190]


def check(precision, shape, zops="tcs", cut=(None, None, None), stride1=False):
    nx, ny, nz = shape
    a = np.random.default_rng(nx * 7 + ny * 3 + nz).standard_normal((nz, ny, nx))
    o = oplan(nx, ny, nz, *cut, stride1=stride1)
    with lib_setup(precision, nx, ny, nz, *cut, stride1=stride1) as P:
        for z in zops:
            if z == "c" and nz < 2:
                continue
            ref = o.ftran_r2c(a, "ff" + z)
            assert rel(P.ftran_r2c(a, "ff" + z), ref) < TOL[precision], (shape, z)
            assert rel(P.btran_c2r(ref, z + "ff"), o.btran_c2r(ref, z + "ff")[0]) < TOL[precision], (shape, z)


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", LENGTHS)
def test_every_axis_and_layout(precision, n):
    check(precision, (n, 5, 6), "t")
    check(precision, (6, n, 5), "t")
    check(precision, (10, 7, n))
    check(precision, (10, 7, n), stride1=True)
    if n > 4:
        c = 2 * (n // 3)
        check(precision, (n, 12, 5), "t", (c, 8, None))
        check(precision, (10, n, n if n < 130 else 15), "t", (6, c, c if n < 130 else 10))
        check(precision, (10, 12, n), "tn", (None, 8, c), stride1=True)


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", LONG)
def test_longest_tiles(precision, n):
    check(precision, (n, 3, 2), "t")
    check(precision, (4, 3, n), "t")
    check(precision, (4, 3, n), "t", stride1=True)


@pytest.mark.parametrize("precision", [8, 4])
def test_more_tiles_than_compute_units(precision):
    """Wide tiles (enough columns for whole 128-byte row segments), a ragged
    last tile, and tiles across plane boundaries."""
    check(precision, (150, 90, 75), "t")
    check(precision, (150, 90, 75), "tc", (100, 60, 50))
    check(precision, (150, 90, 75), "t", stride1=True)
