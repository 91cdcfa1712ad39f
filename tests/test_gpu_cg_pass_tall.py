"""CG in one pass per iteration on the 32-row tiles, which grids with enough planes
take where the last row of tiles is more than half full, and with a set z-chunk
(several planes per chunk and a short last one) on both tile heights; against the
plain numpy CG of the 16-row tests.

FP64: 1e-12 relative max-norm after five iterations, as there.  FP32 (the inner CG
under refinement, three iterations of it): an iteration adds about ten roundings of
2^-24 to a residual whose step is at most a few times as large as it is, and the
directions carry them on, below 1e-4 in all; a wrong ring or tile edge is an error
of the size of the values.
"""
import functools

import numpy as np
import pytest

from tests.test_gpu_cg_pass import apply_a, cg, context

pytestmark = pytest.mark.gpu

TALL = (65, 50, 2050)  # a last tile of one column, a last row of tiles of 18 rows
BCS = [(0, 0, 0, 0, 0, 0), (0, 1, 1, 0, 1, 0)]


def takes_32_rows(n):
    """The pass's rule: two 16-plane chunks of work per compute unit, a last row more than half full."""
    tiles = -(-n[0] // 64) * -(-n[1] // 32)
    return tiles * n[2] >= 2 * 16 * 256 and (n[1] - 1) % 32 + 1 > 16


@functools.lru_cache(maxsize=1)
def reference(n, ds, iters):
    b = np.random.default_rng(sum(n)).normal(size=n[::-1])
    return (b,) + cg(b, ds, iters)


def fp64(C, L, n, ds, sl, deferred, kind):
    b, x, norms = reference(n, ds, 5)
    f = np.zeros(C.shape)
    f[sl] = b
    C.set_deferred_x(deferred)
    C.fill(L.FIELD_X, 0.0)
    C.upload(L.FIELD_B, f)
    res = C.solve([dict(kind=L.CG, tol=0.0, maxit=5), dict(kind=getattr(L, kind))])
    got = C.download(L.FIELD_X)[sl]
    assert np.abs(got - x).max() <= 1e-12 * np.abs(x).max()
    ref = np.array(norms) / np.linalg.norm(b)
    assert np.all(np.abs(res["history"][1:] - ref) <= 1e-11 * ref)


@pytest.mark.parametrize("bcs", BCS)
@pytest.mark.parametrize("deferred,kind", [(True, "NONE"), (False, "JACOBI")])
@pytest.mark.parametrize("kz", [0, 7])
def test_32_row_tiles_match_numpy(kz, deferred, kind, bcs):
    import parallelpoissonsolver_amd._lib as L
    assert takes_32_rows(TALL)
    C, ds, sl = context(L, TALL, bcs)
    C.set_tiling(kz_stencil=kz)
    fp64(C, L, TALL, ds, sl, deferred, kind)
    C.close()


# chunks of 4, 4, 1 and of 6, 6, 5 planes
@pytest.mark.parametrize("n,kz", [((130, 70, 9), 4), ((65, 17, 17), 6)])
@pytest.mark.parametrize("deferred,kind", [(True, "NONE"), (False, "JACOBI")])
def test_set_chunks_match_numpy(n, kz, deferred, kind):
    import parallelpoissonsolver_amd._lib as L
    assert not takes_32_rows(n)
    C, ds, sl = context(L, n, BCS[0])
    C.set_tiling(kz_stencil=kz)
    fp64(C, L, n, ds, sl, deferred, kind)
    C.close()


@pytest.mark.parametrize("deferred", [True, False])
@pytest.mark.parametrize("n,kz", [(TALL, 0), (TALL, 7), ((130, 70, 9), 4)])
def test_fp32_inner_cg_matches_numpy(n, kz, deferred):
    import parallelpoissonsolver_amd._lib as L
    C, ds, sl = context(L, n, BCS[0])
    C.set_tiling(kz_stencil=kz)
    C.set_deferred_x(deferred)
    b, x, _ = reference(n, ds, 3)
    f = np.zeros(C.shape)
    f[sl] = b
    C.fill(L.FIELD_X, 0.0)
    C.upload(L.FIELD_B, f)
    res = C.solve([dict(kind=L.IR, tol=0.0, maxit=1), dict(kind=L.CG, precision=32, tol=0.0, maxit=3),
                   dict(kind=L.NONE, precision=32)])
    assert res["iterations"] == 3
    got = C.download(L.FIELD_X)[sl]
    assert np.abs(got - x).max() <= 1e-4 * np.abs(x).max()
    r = np.linalg.norm(b - apply_a(got, ds)) / np.linalg.norm(b)
    assert abs(res["error_compute_operator"] - r) <= 1e-9 * r
    C.close()
