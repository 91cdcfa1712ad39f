"""Fused Chebyshev sweeps on set z-chunks: a block that marches through several
planes and a short last chunk, on the 16-row tiles (which small grids take with
chunks of one plane) and the 32-row ones, with even and odd numbers of steps.
Against one sweep per launch, with the same bar: 1e-14 (FP64) and 1e-6 (FP32)
relative max-norm.
"""
import numpy as np
import pytest

from tests.test_gpu_cheb_multi import MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [4, 5, 11])  # two, three and three times three levels
@pytest.mark.parametrize("bcs", MIXED)
@pytest.mark.parametrize("n,kz", [((66, 18, 31), 7), ((67, 19, 31), 8), ((130, 64, 550), 9)])
@pytest.mark.parametrize("prec", [64, 32])
def test_set_chunks_match_single_sweeps(n, kz, bcs, m, prec):
    import parallelpoissonsolver_amd._lib as L
    C = L.Context(n, (0.01, 0.012, 0.011), bcs=bcs)
    inp = np.random.default_rng(m).standard_normal(C.shape)
    chain = [dict(kind=L.CHEBYSHEV, precision=prec, maxit=m, cheb_eps=0.0, cheb_rmin=100.0, cheb_rmax=1 - 1e-4)]
    out = {}
    for fused in (1, 0):
        C.set_cheb_pairs(fused, kz)
        C.upload(L.FIELD_T0, inp)
        C.fill(L.FIELD_T1, 0.0)
        assert C.precondition(chain, L.FIELD_T1, L.FIELD_T0) == m
        out[fused] = C.download(L.FIELD_T1)
    C.close()
    diff = np.abs(out[1] - out[0]).max() / np.abs(out[0]).max()
    assert diff <= (1e-14 if prec == 64 else 1e-6), diff
