"""The network's kernels where a block marches through more than one pair of planes.

The z-chunks follow the grid: up to about 96^3 every kernel takes chunks of two
planes, so the small grids of the other tests never reach the interior loops.  The
grids here give the output kernel chunks of 8 planes and the lift chunks of 6, each
with a short last one, and the batches give the convolutions chunks of 6 and 14.
"""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import parallelpoissonsolver_amd._lib as L  # noqa: E402
import tests.test_gpu_nn as N  # noqa: E402
import tests.test_gpu_output_layer as OUT  # noqa: E402
from oracle import nn_oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu

LARGE = (146, 131, 75)  # output kernel 8 planes (3 left over), lift 6 planes (3 left over)


@pytest.fixture(scope="module")
def net():
    n = L.Network(seed=3)
    yield n
    n.close()


def test_output_layer_long_chunks():
    OUT.test_output_layer_tile_edges(LARGE)


def test_fp32_fields_and_gamma_long_chunks(net):
    N.test_fp32_fields_and_fused_gamma(net, LARGE)


@pytest.mark.parametrize("prec", [64, 32])
def test_residual_update_long_chunks(net, prec):
    N.test_fused_residual_update(net, prec, LARGE)


def test_inference_against_the_oracle_long_chunks(net):
    N.test_inference_path_matches_training_forward(net, LARGE)


@pytest.mark.parametrize("batch", [200, 300])
def test_chunks_of_a_batch_do_not_change_a_sample(net, batch):
    """A sample's activations and output are bit for bit the same in a batch, whose
    convolutions run in chunks of 6 (200) or 14 (300) of 25 planes, as alone, where
    they run in chunks of 2."""
    net.set_params(N._params(41))
    x = np.random.default_rng(42).normal(size=(batch, 50, 32, 32)).astype(np.float32)
    y = net.forward(x)
    acts = {i: net.activation(i) for i in (2, 10, 12)}
    for k in (0, batch // 2, batch - 1):
        alone = net.forward(x[k:k + 1])
        assert np.array_equal(alone[0], y[k])
        for i, a in acts.items():
            assert np.array_equal(net.activation(i)[0], a[k]), i


def reach(n, v, lift):
    """Points of a line of n that a single input point v can change, layer by layer
    (lift: the first layer's reach, in points)."""
    def grow(m, r):
        out = m.copy()
        for d in range(1, r + 1):
            out[d:] |= m[:-d]
            out[:-d] |= m[d:]
        return out

    def pool(m):
        return np.pad(m, (0, m.size % 2)).reshape(-1, 2).any(axis=1)

    src = np.zeros(n, bool)
    src[v] = True
    acts = []
    for cin, cout, level, mode, ia, sk, relu in O.NET:
        if mode == "field":
            acts.append(grow(src, lift))
            continue
        m = acts[ia]
        if mode == "pool":
            m = pool(m)
        elif mode == "upadd":
            m = m.repeat(2)[:acts[sk].size] | acts[sk]
        acts.append(grow(m, 1))
    # the output layer recomputes the lift: its skip is as wide as activation 0
    return acts[-1]


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("prec", [64, 32])
def test_a_non_finite_voxel_stays_in_its_neighbourhood(net, prec, bad):
    """The output kernel keeps the sums of four planes in slots, one of them idle on
    each plane; a non-finite plane must not leak through the idle slot.  Outputs that
    the voxel cannot reach are those of the clean input, bit for bit.  In x and y the
    first layer's operands also hold a column with zero weights one voxel further out
    (0 times infinity is NaN), so its reach counts as 2 there.  What an infinity does
    reach is not finite; a NaN may end in the first ReLU, which takes the larger of
    its bits and 0 and so returns 0 for a NaN with the sign bit set."""
    nx, ny, nz = dims = (98, 90, 150)
    v = (12, 9, 60)
    net.set_params(N._params(43))
    C = L.Context(tuple(d + 2 for d in dims), tuple(1.0 / (d + 1) for d in dims))
    net.attach(C)
    inside = (slice(2, -2),) * 3
    f = np.zeros(C.shape)
    f[inside] = np.random.default_rng(44).choice([-1.0, 1.0], size=(nz, ny, nx))
    C.fill(L.FIELD_T2, 0.0)
    out = {}
    for name in ("clean", "bad"):
        if name == "bad":
            f[2 + v[2], 2 + v[1], 2 + v[0]] = bad
        C.upload(L.FIELD_T0, f)
        C.fill(L.FIELD_X, 0.0)
        C.fill(L.FIELD_T1, 0.0)
        C.nn_apply_update(L.FIELD_T1, L.FIELD_T0, L.FIELD_T2, L.FIELD_X, 0.0, float(nx * ny * nz), prec=prec)
        out[name] = C.download(L.FIELD_T1)[inside]
    C.close()
    rx, ry, rz = reach(nx, v[0], 2), reach(ny, v[1], 2), reach(nz, v[2], 1)
    touched = rz[:, None, None] & ry[None, :, None] & rx[None, None, :]
    assert np.isfinite(out["clean"]).all()
    assert 10 < (~rz).sum() and (~rx).sum() > 10
    assert np.array_equal(out["bad"][~touched], out["clean"][~touched])
    if np.isinf(bad):
        assert not np.isfinite(out["bad"][v[2], v[1], v[0]])
