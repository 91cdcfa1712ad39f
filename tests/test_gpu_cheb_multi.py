"""Fused Chebyshev sweeps (two and three per pass, the first pass with the
recurrence's start) against one sweep per launch, where the tiles of 64 x 16 and
64 x 32 points end: one point short of, exactly at and one past a tile, a last
row of tiles that is half full, grids with enough planes for the taller tiles.
Both paths evaluate the same expressions, so the bar is rounding level: 1e-14
(FP64) and 1e-6 (FP32) relative max-norm.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# data points; the last two have 32-row tiles (6 x 348 and 4 x 548 tile-planes of 2048)
SIZES = [(65, 17, 5), (66, 18, 4), (67, 19, 9), (131, 51, 350), (130, 64, 550)]
MIXED = [(0, 0, 0, 0, 0, 0), (0, 1, 1, 0, 1, 0), (1, 0, 0, 1, 0, 1)]


@pytest.mark.parametrize("m", [4, 5, 6, 11])  # 2, 3, 2+2 and 3+3+3 levels
@pytest.mark.parametrize("bcs", MIXED)
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("prec", [64, 32])
def test_fused_sweeps_match_single_sweeps(n, bcs, m, prec):
    import parallelpoissonsolver_amd._lib as L
    C = L.Context(n, (0.01, 0.012, 0.011), bcs=bcs)
    inp = np.random.default_rng(m).standard_normal(C.shape)
    chain = [dict(kind=L.CHEBYSHEV, precision=prec, maxit=m, cheb_eps=0.0, cheb_rmin=100.0, cheb_rmax=1 - 1e-4)]
    out = {}
    for fused in (1, 0):
        C.set_cheb_pairs(fused)
        C.upload(L.FIELD_T0, inp)
        C.fill(L.FIELD_T1, 0.0)
        assert C.precondition(chain, L.FIELD_T1, L.FIELD_T0) == m
        out[fused] = C.download(L.FIELD_T1)
    C.close()
    diff = np.abs(out[1] - out[0]).max() / np.abs(out[0]).max()
    assert diff <= (1e-14 if prec == 64 else 1e-6), diff
