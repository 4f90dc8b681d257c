"""The specialised X tiles (in-place stages, first stage from and last stage
to memory) and the plane kernels built on them, against the FP64 oracle: every
specialised length, ragged and odd numbers of rows, one row, X cuts, and every
plane shape.  Tolerances as test_gpu_parity.py."""
import numpy as np
import pytest

import p3dfft_amd
from test_gpu_parity import TOL, lib_setup, oplan, rel

pytestmark = pytest.mark.gpu

LENS = (32, 48, 64, 96, 128, 160, 192, 256, 320, 384, 512, 1024, 2048)
CASES = [((n, 5, 7), None) for n in LENS] + [((n, 1, 1), None) for n in (48, 64, 512, 2048)]
CASES += [((96, 9, 4), (64, None, None)), ((384, 6, 11), (256, None, None)), ((2048, 3, 3), (2, None, None))]
PLANES = [(32, 32, 3), (64, 64, 5), (32, 64, 2), (64, 32, 4), (128, 64, 3), (64, 128, 2), (128, 128, 2)]


def check(precision, n, cut, seed):
    nx, ny, nz = n
    cut = cut or (None, None, None)
    a = np.random.default_rng(seed).standard_normal((nz, ny, nx))
    o = oplan(nx, ny, nz, *cut)
    ref = o.ftran_r2c(a)
    with lib_setup(precision, nx, ny, nz, *cut) as P:
        assert rel(P.ftran_r2c(a), ref) < TOL[precision]
        assert rel(P.btran_c2r(ref, "tff"), o.btran_c2r(ref, "tff")[0]) < TOL[precision]


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_x_tile_against_oracle(precision, k):
    check(precision, *CASES[k], k)


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", PLANES)
def test_plane_against_oracle(precision, n):
    lib = p3dfft_amd.load(precision)
    lib.p3dfft_amd_set_plane_kernels(1)
    try:
        check(precision, n, None, sum(n))
    finally:
        lib.p3dfft_amd_set_plane_kernels(2)
