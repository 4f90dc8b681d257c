"""The persistent 2048-point column kernel: more tiles than workgroups with a
narrow last round, peers with equal blocks (separable rows), unequal ones (row
tables) and cut rows (some missing).  Tolerances as test_gpu_parity.py."""
import numpy as np
import pytest

import p3dfft_amd
from oracle import oracle as O
from test_gpu_parity import TOL, lib_setup, oplan, rel
from test_gpu_share import run_grid_on_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", [(34, 116, 2048), (34, 2048, 115)])
def test_narrow_last_round(precision, n):
    """18 x 116 (115) columns: one or two rounds of the CUs, then 40 (22) columns"""
    nx, ny, nz = n
    a = np.random.default_rng(nz).standard_normal((nz, ny, nx))
    ref = np.fft.rfftn(a)
    with lib_setup(precision, nx, ny, nz) as P:
        s = P.ftran_r2c(a)
        assert rel(s, ref) < TOL[precision]
        assert rel(P.btran_c2r(s, "tff"), a * nx * ny * nz) < TOL[precision] * 10


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("n", [(34, 47, 2048), (34, 2048, 200), (34, 200, 2048), (2, 1, 2048)])
def test_full_last_round(precision, n):
    """846 columns (no whole round), 3600 (a remainder of three quarters of a round
    and more) and 2: full tiles, the last one partial"""
    nx, ny, nz = n
    a = np.random.default_rng(ny).standard_normal((nz, ny, nx))
    ref = np.fft.rfftn(a)
    with lib_setup(precision, nx, ny, nz) as P:
        s = P.ftran_r2c(a)
        assert rel(s, ref) < TOL[precision]
        assert rel(P.btran_c2r(s, "tff"), a * nx * ny * nz) < TOL[precision] * 10


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("dims", [(2, 4), (3, 2)])
def test_peer_blocks(precision, dims):
    nx, ny, nz = 18, 2048, 16
    a = np.random.default_rng(11).standard_normal((nz, ny, nx))
    spec, field, _ = run_grid_on_gpu(precision, dims, nx, ny, nz, a)
    full = O.Plan(nx, ny, nz).ftran_r2c(a)
    for (i, j), s in spec.items():
        o = O.Plan(nx, ny, nz, dims=dims, ipid=i, jpid=j)
        ref = full[:, o.jjstart - 1:o.jjend, o.iistart - 1:o.iiend].reshape(-1)
        assert rel(s, ref) < TOL[precision], (i, j)
    assert rel(field, a * nx * ny * nz) < TOL[precision] * 10


@pytest.mark.parametrize("precision", [8, 4])
def test_cut_rows(precision):
    """Rows of the padded length missing: equal to the separate pack passes"""
    dims, n, cut = (2, 2), (18, 2048, 16), (12, 1366, 12)
    S = p3dfft_amd.Share(precision)
    rng = np.random.default_rng(13)
    S.setup_share(dims, 1, 1, *n, *cut)
    try:
        for fn, nin, nout in ((S.ftran_y, S.n_ypen(), S.n_send2()), (S.btran_y, S.n_send2(), S.n_ypen())):
            x = (rng.standard_normal(nin) + 1j * rng.standard_normal(nin)).astype(S.cdtype)
            got = []
            for fused in (1, 0):
                S.lib.p3dfft_share_set_fused(fused)
                a, b = S.alloc(x.nbytes), S.alloc(nout * x.itemsize)
                a.upload(x)
                b.upload(np.zeros(nout, dtype=S.cdtype))
                fn(a, b)
                got.append(b.download(nout, S.cdtype).astype(np.complex128))
                a.free()
                b.free()
            assert rel(got[0], got[1]) < TOL[precision] / 10
    finally:
        S.lib.p3dfft_share_set_fused(1)
        S.clean()
