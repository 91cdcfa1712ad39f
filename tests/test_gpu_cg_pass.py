"""CG in one pass per iteration (pointwise preconditioners) against a plain
numpy CG, at the edges of its tiles and chunks.

The pass forms r_k, p_k and A p_k from r_{k-1} and p_{k-1} and predicts
||r_{k+1}||; a step that removes most of the residual is followed by a pass that
recomputes it.  After a few iterations from one right-hand side the two differ
by rounding only, far below the 1e-12 relative max-norm asked for here.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# interior points: a single one, one short of / exactly / one past a tile in
# each direction, several tiles; the last one takes the 32-row tiles (enough
# 16-plane chunks for two per CU)
SIZES = [(1, 1, 1), (63, 15, 5), (64, 16, 17), (65, 17, 6), (130, 70, 9), (65, 33, 2050)]


def apply_a(p, ds):
    """The 7-point operator on the solver region, zero around it."""
    q = np.pad(p, 1)
    c = [1.0 / (d * d) for d in ds]
    out = -2.0 * (c[0] + c[1] + c[2]) * p
    out += c[0] * (q[1:-1, 1:-1, :-2] + q[1:-1, 1:-1, 2:])
    out += c[1] * (q[1:-1, :-2, 1:-1] + q[1:-1, 2:, 1:-1])
    out += c[2] * (q[:-2, 1:-1, 1:-1] + q[2:, 1:-1, 1:-1])
    return out


def cg(b, ds, iters):
    x, r = np.zeros_like(b), b.copy()
    p, rr = np.zeros_like(b), float((b * b).sum())
    beta = 0.0
    norms = []
    for _ in range(iters):
        p = r + beta * p
        ap = apply_a(p, ds)
        a = rr / float((p * ap).sum())
        x += a * p
        r -= a * ap
        new = float((r * r).sum())
        beta, rr = new / rr, new
        norms.append(np.sqrt(new))
    return x, norms


def context(L, n, bcs):
    """Context whose solver region has n points, and that region's slice of a guarded field."""
    npg = [n[d] + (bcs[2 * d] == 0) + (bcs[2 * d + 1] == 0) for d in range(3)]
    ds = (0.01, 0.0125, 0.011)
    C = L.Context(npg, ds, bcs=bcs)
    lo = [1 + (bcs[2 * d] == 0) for d in range(3)]
    return C, ds, tuple(slice(lo[d], lo[d] + n[d]) for d in (2, 1, 0))


@pytest.mark.parametrize("bcs", [(0, 0, 0, 0, 0, 0), (0, 1, 1, 0, 1, 0)])
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("deferred,kind", [(True, "NONE"), (False, "JACOBI")])
def test_one_pass_cg_matches_numpy(n, bcs, deferred, kind):
    import parallelpoissonsolver_amd._lib as L
    if min(npg_of(n, bcs)) < 3:
        n = (max(n[0], 2), max(n[1], 2), max(n[2], 2))
    C, ds, sl = context(L, n, bcs)
    b = np.zeros(C.shape)
    b[sl] = np.random.default_rng(sum(n)).normal(size=b[sl].shape)
    C.set_deferred_x(deferred)
    single = n == (1, 1, 1)
    for iters in ([1] if min(n) == 1 or max(n) <= 2 else [1, 5]):
        C.fill(L.FIELD_X, 0.0)
        C.upload(L.FIELD_B, b)
        res = C.solve([dict(kind=L.CG, tol=1e-13 if single else 0.0, maxit=iters + (5 if single else 0)),
                       dict(kind=getattr(L, kind))])
        x, norms = cg(b[sl], ds, iters)
        got = C.download(L.FIELD_X)[sl]
        assert res["iterations"] == iters
        assert np.abs(got - x).max() <= 1e-12 * np.abs(x).max()
        if not single:
            ref = np.array(norms) / np.linalg.norm(b[sl])
            assert np.all(np.abs(res["history"][1:] - ref) <= 1e-11 * ref)
    C.close()


def npg_of(n, bcs):
    return [n[d] + (bcs[2 * d] == 0) + (bcs[2 * d + 1] == 0) for d in range(3)]


@pytest.mark.parametrize("deferred", [True, False])
def test_a_step_that_removes_the_residual_is_recomputed(deferred):
    """A discrete sine is an eigenvector: one iteration, whose residual the
    prediction cannot resolve (it cancels to ~1e-16 of ||r||^2); with a second,
    smaller mode the loop goes on from the recomputed residual."""
    import parallelpoissonsolver_amd._lib as L
    n = (33, 20, 18)
    C, ds, sl = context(L, n, (0, 0, 0, 0, 0, 0))
    C.set_deferred_x(deferred)

    def mode(kx, ky, kz):
        f = [np.sin(k * np.pi * np.arange(1, m + 1) / (m + 1)) for k, m in zip((kx, ky, kz), n)]
        return f[2][:, None, None] * f[1][None, :, None] * f[0][None, None, :]

    for rhs, most in ((mode(1, 1, 1), 1), (mode(1, 1, 1) + 1e-6 * mode(5, 3, 2), 3)):
        b = np.zeros(C.shape)
        b[sl] = rhs
        C.fill(L.FIELD_X, 0.0)
        C.upload(L.FIELD_B, b)
        res = C.solve([dict(kind=L.CG, tol=1e-11, maxit=50), dict(kind=L.NONE)])
        assert res["iterations"] <= most
        assert res["error_compute_operator"] < 1e-11
        assert res["error_from_iteration"] == res["history"][res["iterations"]]
        assert res["error_from_iteration"] < 1e-11
    C.close()


@pytest.mark.parametrize("n", [(65, 17, 6), (65, 33, 2050)])
def test_one_pass_fp32_inner_cg(n):
    """The FP32 form under FP64 refinement reaches an FP64 residual."""
    import parallelpoissonsolver_amd._lib as L
    C, ds, sl = context(L, n, (0, 0, 0, 0, 0, 0))
    b = np.zeros(C.shape)
    b[sl] = np.random.default_rng(1).normal(size=b[sl].shape)
    C.fill(L.FIELD_X, 0.0)
    C.upload(L.FIELD_B, b)
    res = C.solve([dict(kind=L.IR, tol=1e-12, maxit=50), dict(kind=L.CG, precision=32, tol=1e-4, maxit=2000),
                   dict(kind=L.NONE, precision=32)])
    x = C.download(L.FIELD_X)[sl]
    assert np.linalg.norm(b[sl] - apply_a(x, ds)) < 1.1e-12 * np.linalg.norm(b[sl])
    assert res["outer_iterations"] <= 6
    C.close()


@pytest.mark.parametrize("deferred", [True, False])
def test_iterations_past_an_exact_solution_stay_finite(deferred):
    """tol = 0 on a grid whose residual underflows to zero before maxit."""
    import parallelpoissonsolver_amd._lib as L
    n = (6, 5, 4)
    C, ds, sl = context(L, n, (0, 0, 0, 0, 0, 0))
    C.set_deferred_x(deferred)
    b = np.zeros(C.shape)
    b[sl] = np.random.default_rng(3).normal(size=b[sl].shape)
    C.fill(L.FIELD_X, 0.0)
    C.upload(L.FIELD_B, b)
    C.solve([dict(kind=L.IR, tol=1e-12, maxit=30),
             dict(kind=L.CG, tol=0.0, maxit=400, precision=32), dict(kind=L.NONE)])
    got = C.download(L.FIELD_X)[sl]
    C.close()
    r = b[sl] - apply_a(got, ds)
    assert np.linalg.norm(r) <= 1e-10 * np.linalg.norm(b[sl])
