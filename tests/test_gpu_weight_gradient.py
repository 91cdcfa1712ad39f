"""The weight-gradient kernel at the edges of its 16 x 16 tiles and z-chunks:
odd extents, one voxel past a tile, single planes at the coarsest level, and a
depth of several chunks.  Against the numpy oracle with the bars of the network's
gradient test: 3 % relative L2 per layer plus half the distance between the
oracle's rounded and exact gradients (what BF16 storage alone moves).
"""
import numpy as np
import pytest

from oracle import nn_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 3, 2, 5), (2, 5, 17, 16), (1, 33, 15, 34), (1, 40, 33, 9)])
def test_weight_gradient_edges(shape):
    import parallelpoissonsolver_amd._lib as L
    net = L.Network(seed=3)
    rng = np.random.default_rng(sum(shape))
    p = O.init_params(5)
    for l in range(O.N_LAYERS):
        p[l * O.LAYER_PARAMS + O.TAPS * 256:(l + 1) * O.LAYER_PARAMS] = rng.normal(0, 0.05, 16)
    net.set_params(p)
    p = net.get_params()
    x = rng.normal(size=shape).astype(np.float32)
    g = rng.uniform(1.0, 3.0, shape[0])
    loss, grad = net.loss_grad(x, g)
    lo, go = O.loss_grad(p, x, g, rounding=True)
    _, gx = O.loss_grad(p.astype(np.float64), x.astype(np.float64), g, rounding=False)
    assert abs(loss - lo) < 1e-3 * max(1.0, abs(lo))
    for l in range(O.N_LAYERS):
        sl = slice(l * O.LAYER_PARAMS, (l + 1) * O.LAYER_PARAMS)
        bf16_effect = np.linalg.norm(go[sl] - gx[sl])
        assert np.linalg.norm(grad[sl] - go[sl]) <= 3e-2 * np.linalg.norm(go[sl]) + 0.5 * bf16_effect + 1e-9, l
    net.close()
