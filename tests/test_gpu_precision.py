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
