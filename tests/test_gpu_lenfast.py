"""The length-fastest (STRIDE1) Z pass of the specialised lengths against the
FP64 oracle: every specialised length (one tile width each), a ragged last
tile, tiles that cross rows of the spectrum, cuts on the length-fastest side,
and more tiles than compute units.  Tolerances as test_gpu_parity.py."""
import numpy as np
import pytest

from test_gpu_parity import TOL, lib_setup, oplan, rel

pytestmark = pytest.mark.gpu

CASES = [((10, 7, n), None) for n in (32, 48, 64, 96, 128, 160, 192, 256, 320, 384, 512, 1024, 2048)]
CASES += [((2, 1, 64), None), ((34, 9, 128), (None, None, 80)), ((34, 9, 512), (20, 6, 3)), ((62, 40, 96), None),
          ((254, 90, 64), (None, None, 42)), ((6, 5, 2048), (None, None, 1366))]


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_lenfast_against_oracle(precision, k):
    (nx, ny, nz), cut = CASES[k]
    cut = cut or (None, None, None)
    a = np.random.default_rng(k).standard_normal((nz, ny, nx))
    o = oplan(nx, ny, nz, *cut, stride1=True)
    ref = o.ftran_r2c(a)
    with lib_setup(precision, nx, ny, nz, *cut, stride1=True) as P:
        assert rel(P.ftran_r2c(a), ref) < TOL[precision]
        assert rel(P.btran_c2r(ref, "tff"), o.btran_c2r(ref, "tff")[0]) < TOL[precision]
