"""The chunk rules of the marching kernels count the device's own compute units."""
from tests import fakehip

CHILD = r"""
fake.fake_cus({cus})
C = L.Context((66, 66, 66), (0.1, 0.1, 0.1))
for k in (L.K_CG_PASS, L.K_CHEB_TRIPLE):
    fake.fake_reset()
    C.time_kernel(k, 1)
    print(fake.fake_blocks())
"""


def test_blocks_follow_the_compute_units(tmp_path):
    """64^3 points: 4 tiles of 16 rows.  256 units: chunks of one plane, a block per unit.
    32 units: longer chunks, since past two blocks per unit more of them only add halo planes."""
    wide = [int(v) for v in fakehip.run(tmp_path, CHILD.format(cus=256)).split()]
    few = [int(v) for v in fakehip.run(tmp_path, CHILD.format(cus=32)).split()]
    assert wide == [256, 256]
    assert all(0 < v <= 2 * 32 for v in few)
