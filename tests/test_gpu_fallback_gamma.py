"""GPU tests of the sums that the learned preconditioner's fallback forms in its
update kernel: one partial per block, 256 points a block up to 2048 blocks."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import parallelpoissonsolver_amd._lib as L  # noqa: E402
from oracle import nn_oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(4, 5, 6), (17, 9, 33), (66, 40, 70), (128, 80, 70)])
def test_fallback_is_jacobi_fcg(dims):
    """A network that returns NaN: the first step is discarded and Jacobi-FCG runs from
    the same residual, so it takes one iteration more than Jacobi-FCG itself.  The
    norms behind the two convergence tests come from different sums: one iteration
    either way.  Wrong partial sums would cost conjugacy and many iterations.  Two
    solutions with residuals of 1e-10 differ by at most cond(A) 2e-10, below 1e4 times
    that on these grids."""
    print(f"[nn] fallback {dims}", flush=True)
    net = L.Network(seed=9)
    p = net.get_params()
    p[13 * O.LAYER_PARAMS + O.TAPS * 256] = np.nan  # output bias -> every output NaN
    net.set_params(p)
    n = tuple(d + 2 for d in dims)
    C = L.Context(n, (1.0 / (max(n) - 1),) * 3)
    net.attach(C)
    b = np.zeros(C.shape)
    b[2:-2, 2:-2, 2:-2] = np.random.default_rng(sum(dims)).normal(size=dims[::-1])
    out = []
    for pre in (dict(kind=L.NN), dict(kind=L.JACOBI)):
        C.upload(L.FIELD_B, b)
        C.fill(L.FIELD_X, 0.0)
        r = C.solve([dict(kind=L.FCG, tol=1e-10, maxit=5000), pre])
        out.append((r["iterations"], C.download(L.FIELD_X)))
    assert abs(out[0][0] - out[1][0] - 1) <= 1
    assert np.linalg.norm(out[0][1] - out[1][1]) < 2e-6 * np.linalg.norm(out[1][1])
    C.close()
    net.close()
