"""Host arrays in and out of device fields: pageable memory goes through dense
blocks of planes on the device, pinned memory through one pitched copy; both
must move every guarded value unchanged."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one row per wavefront and fewer rows than a block, a ragged box, rows longer
# than a wavefront, and a field of several 64 MiB blocks with a short last one
SHAPES = [(3, 3, 3), (63, 5, 4), (131, 35, 43), (700, 3, 9), (258, 258, 150)]


@pytest.mark.parametrize("n", SHAPES)
def test_pageable_and_pinned_transfers_agree(n):
    import torch

    import parallelpoissonsolver_amd._lib as L
    C = L.Context(n, (0.1, 0.2, 0.3))
    rng = np.random.default_rng(sum(n))
    a = rng.normal(size=C.shape)
    pinned = torch.empty(C.shape, dtype=torch.float64, pin_memory=True)
    ptr = ctypes.cast(pinned.data_ptr(), ctypes.POINTER(ctypes.c_double))
    C.upload(L.FIELD_T0, a)
    C._chk(L.lib().pps_download(C.h, L.FIELD_T0, ptr))
    assert np.array_equal(pinned.numpy(), a)
    pinned.copy_(torch.from_numpy(-2.0 * a))
    C._chk(L.lib().pps_upload(C.h, L.FIELD_T1, ptr))
    assert np.array_equal(C.download(L.FIELD_T1), -2.0 * a)
    assert np.array_equal(C.download(L.FIELD_T0), a)
    C.close()
