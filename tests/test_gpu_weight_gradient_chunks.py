"""The weight-gradient kernel where a block marches through several planes.

Its z-chunks give every compute unit three blocks, so on small batches each block
takes one plane and never turns its ring of staged planes.  Here one sample is one
tile (or four) and the batch is large: chunks of 6, 3 and 2 planes at the three
levels with short last ones (batch 200), and of 9 at level 0 (batch 60).  Same bar
as on the small batches: 1.5 % per layer, where a lost plane is 3 % of the voxels
or more.
"""
import pytest

from tests import test_gpu_weight_gradient as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(200, 21, 6, 7), (60, 33, 18, 20)])
def test_weight_gradient_long_chunks(shape):
    W.test_weight_gradient_edges(shape)
