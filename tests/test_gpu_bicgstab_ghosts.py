"""BiCGSTAB's two operator applications form the Neumann ghosts of their input
themselves: against a plain numpy BiCGSTAB with mirrored ghosts, where the faces
meet the edges of the 64 x 16 tiles and of the z-chunks.  A wrong ghost is an
error of order one; rounding after four iterations from a random right-hand side
is below 1e-12, the bar 1e-10 of the max-norm.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# points of the solver region
SIZES = [(3, 2, 2), (63, 15, 3), (64, 16, 17), (65, 17, 6), (130, 33, 40)]
BCS = [(1, 0, 0, 1, 0, 1), (0, 1, 1, 0, 1, 0), (1, 1, 0, 1, 1, 0)]


def apply_a(p, ds, bcs):
    q = np.pad(p, 1)
    # ghost beyond a Neumann face = the point two cells inward
    for axis, d in ((2, 0), (1, 1), (0, 2)):
        v = np.moveaxis(q, axis, 0)
        if bcs[2 * d]:
            v[0] = v[2]
        if bcs[2 * d + 1]:
            v[-1] = v[-3]
    c = [1.0 / (d * d) for d in ds]
    out = -2.0 * (c[0] + c[1] + c[2]) * p
    out += c[0] * (q[1:-1, 1:-1, :-2] + q[1:-1, 1:-1, 2:])
    out += c[1] * (q[1:-1, :-2, 1:-1] + q[1:-1, 2:, 1:-1])
    out += c[2] * (q[:-2, 1:-1, 1:-1] + q[2:, 1:-1, 1:-1])
    return out


def bicgstab(b, ds, bcs, iters):
    x, r, r0, p = np.zeros_like(b), b.copy(), b.copy(), b.copy()
    rho = float((r * r0).sum())
    for _ in range(iters):
        ap = apply_a(p, ds, bcs)
        a = rho / float((ap * r0).sum())
        r = r - a * ap
        ar = apply_a(r, ds, bcs)
        w = float((ar * r).sum()) / float((ar * ar).sum())
        x += a * p + w * r
        r = r - w * ar
        new = float((r * r0).sum())
        p = r + new / rho * a / w * (p - w * ap)
        rho = new
    return x


@pytest.mark.parametrize("bcs", BCS)
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("kind", ["NONE", "JACOBI"])
def test_mirrored_ghosts(n, bcs, kind):
    import parallelpoissonsolver_amd._lib as L
    npg = [n[d] + (bcs[2 * d] == 0) + (bcs[2 * d + 1] == 0) for d in range(3)]
    ds = (0.01, 0.0125, 0.011)
    C = L.Context(npg, ds, bcs=bcs)
    lo = [1 + (bcs[2 * d] == 0) for d in range(3)]
    sl = tuple(slice(lo[d], lo[d] + n[d]) for d in (2, 1, 0))
    b = np.zeros(C.shape)
    b[sl] = np.random.default_rng(sum(n)).normal(size=b[sl].shape)
    iters = 2 if max(n) == 3 else 4
    C.fill(L.FIELD_X, 0.0)
    C.upload(L.FIELD_B, b)
    C.solve([dict(kind=L.BICGSTAB, tol=0.0, maxit=iters), dict(kind=getattr(L, kind))])
    got = C.download(L.FIELD_X)[sl]
    C.close()
    x = bicgstab(b[sl], ds, bcs, iters)
    assert np.abs(got - x).max() <= 1e-10 * np.abs(x).max()
