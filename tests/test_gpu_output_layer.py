"""GPU tests of the fused output layer at the edges of its tiles (14 x 16 voxels,
wavefronts of 4 rows), of its slots in z (four planes) and of its z-chunks."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import parallelpoissonsolver_amd._lib as L  # noqa: E402
from oracle import nn_oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(14, 16, 4), (15, 17, 5), (13, 15, 6), (28, 33, 7), (29, 31, 2), (43, 50, 9),
                                  (3, 4, 3), (17, 48, 67)])
def test_output_layer_tile_edges(dims):
    """The solver's path on random signs (RMS 1, so both paths stage the same input)
    against the oracle's output layer on the GPU's own activations.  The BF16
    products are exact in FP32 and 27 x 32 of them are added in FP32: 2e-5 in L2, and
    per voxel 864 roundings of partial sums below 8 times the largest output,
    864 * 8 * 2^-24 < 5e-4 of it."""
    nx, ny, nz = dims
    print(f"[nn] output layer {dims}", flush=True)
    net = L.Network(seed=5)
    C = L.Context((nx + 2, ny + 2, nz + 2), (1.0 / (nx + 1), 1.0 / (ny + 1), 1.0 / (nz + 1)))
    net.attach(C)
    p = net.get_params()
    r = np.random.default_rng(nx + ny + nz).choice([-1.0, 1.0], size=(nz, ny, nx))
    f = np.zeros(C.shape)
    f[2:-2, 2:-2, 2:-2] = r
    C.upload(L.FIELD_T0, f)
    C.fill(L.FIELD_T1, 0.0)
    C.nn_apply(L.FIELD_T1, L.FIELD_T0)
    out = C.download(L.FIELD_T1)
    y = out[2:-2, 2:-2, 2:-2].copy()
    out[2:-2, 2:-2, 2:-2] = 0.0
    assert not out.any()  # nothing is written outside the region
    net.forward(r[None].astype(np.float32))
    want = O.output_layer(p, net.activation(0), net.activation(12), exact_skip=True)[0]
    assert np.linalg.norm(y - want) < 2e-5 * np.linalg.norm(want)
    assert np.max(np.abs(y - want)) < 5e-4 * np.max(np.abs(want))
    C.close()
    net.close()
