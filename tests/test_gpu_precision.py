"""FP32 accuracy that the relative errors of a single pass do not show: the
constants of the butterflies."""
import numpy as np
import pytest

from test_gpu_parity import lib_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [9, 81])
def test_ninth_roots_are_rounded_once(n):
    """An impulse at the second value of a radix-9 butterfly gives A W9^k at the
    outputs k = 1, 2 (mod 9): the stage twiddles hold hi + lo, and so does W9, so
    each component is the exact product rounded once, within half an ulp (and
    2^-25 of one, the rounding of the lo term).  X has two points, which are exact
    sums."""
    m = 4096
    amp = np.random.default_rng(n).uniform(1, 2, m).astype(np.float32)
    a = np.zeros((m, n, 2), dtype=np.float32)
    a[:, n // 9, 0] = amp
    with lib_setup(4, 2, n, m) as P:
        s = P.ftran_r2c(a, "ffn")
    for k in (1, 2):
        w = np.exp(-2j * np.pi * k / 9)
        for part, c in ((s.real, w.real), (s.imag, w.imag)):
            got = part[:, k::9, 0].astype(np.float64)
            exact = amp.astype(np.float64)[:, None] * c
            ulp = np.spacing(np.abs(exact).astype(np.float32)).astype(np.float64)
            assert (np.abs(got - exact) <= (0.5 + 1e-6) * ulp).all(), k


def test_384_points_keep_the_mean_amplitude():
    """A forward and a backward transform with butterfly constants rounded to
    FP32 scale white noise by a small constant, which adds up over the axes of a
    box, unlike rounding.  One radix 8 (a quarter of the energy passes a product
    with sqrt(1/2) each way) and one radix 3 (a third, with sqrt(3)/2) scale it by
    -2.05e-8; another radix 8 would make it -2.9e-8.  Rounding leaves the mean of
    2^20 values uncertain by about 1.5e-10."""
    n, m = 384, 1 << 11
    e8 = float(np.float32(np.sqrt(0.5))) / np.sqrt(0.5) - 1
    e3 = float(np.float32(np.sqrt(0.75))) / np.sqrt(0.75) - 1
    bound = abs(2 * (e8 / 4 + e3 / 3)) + 1e-9
    a = np.random.default_rng(1).standard_normal((m, n, 2)).astype(np.float32)
    with lib_setup(4, 2, n, m) as P:
        b = P.btran_c2r(P.ftran_r2c(a, "ffn"), "nff").astype(np.float64) / (2 * n)
    x = a.astype(np.float64)
    assert abs((x * (b - x)).sum() / (x * x).sum()) < bound
